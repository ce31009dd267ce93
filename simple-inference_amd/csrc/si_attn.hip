// si_attn.hip -- RoPE + fp16 K/V append, and GQA attention over the fp16
// cache for decode, batched decode and causal prefill.
//
// RoPE (qwen_one_layer.c:172-183) uses cos/sin tables computed on the host
// with the reference's libm calls (as register_fusion.h:364-369 does), so
// the rotation  a' = a*c - b*s,  b' = b*c + a*s  and the fp16 narrowing of
// the new K/V rows are bit-exact given identical projections.
//
// Attention (attention_flash, attention_kernels.h:80-164) is split over the
// context ("flash-decoding"): each workgroup owns one query, one KV group
// (all qheads/kvheads query heads that share it, so every K/V byte is read
// once per query) and one context chunk, runs the scores and the weighted
// V sum on the fp16 matrix cores with an online softmax, and leaves
// (max, sum, unnormalised output) partials; a second kernel merges the
// chunks, normalises and quantizes the result to Q8_0 (the reference's next
// step, qwen_one_layer.c:272).
#include "si_device.hpp"
#include "si_kernels.hpp"

namespace si {

// grid (ntok, ceil((qheads + kvheads) * hdim/2 / 256)), block 256: one
// thread per rotation pair (head h = j / (hdim/2), pair i = j % (hdim/2) of
// token t), so a workgroup covers several heads of a token (half-wavefront
// workgroups per head had left most lanes idle).  With a page table
// (pg.pages != nullptr) token t's K/V row goes to the pool row of sequence
// t's position pos (kv_seq_stride unused).
constexpr int ROPE_T = 256;
__global__ void __launch_bounds__(ROPE_T) k_rope_kv(
    const float *__restrict__ qkv, int ldqkv, int qheads, int kvheads, int hdim, int pos0,
    int pos_step, int max_pos, const int *__restrict__ ctx_dev, const float *__restrict__ rc,
    const float *__restrict__ rs, float *__restrict__ q_out, uint16_t *__restrict__ kc,
    uint16_t *__restrict__ vc, size_t kv_seq_stride, KvPages pg) {
    const int t = blockIdx.x;
    const int half = hdim >> 1;
    const int j = blockIdx.y * ROPE_T + threadIdx.x;
    if (j >= (qheads + kvheads) * half) return;
    const int h = j / half, i = j - h * half;
    const int pos = ctx_dev ? ctx_dev[t] - 1 : pos0 + t * pos_step;
    if (pos < 0 || pos >= max_pos) return;  // device-supplied contexts are not host-checked
    const float c = rc[(size_t)pos * half + i], s = rs[(size_t)pos * half + i];
    const float *row = qkv + (size_t)t * ldqkv;
    const int qd = qheads * hdim, kvd = kvheads * hdim;
    if (h < qheads) {
        const float a = row[h * hdim + i], b = row[h * hdim + i + half];
        float *qo = q_out + (size_t)t * qd + h * hdim;
        qo[i] = __fsub_rn(__fmul_rn(a, c), __fmul_rn(b, s));
        qo[i + half] = __fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s));
    } else {
        const int g = h - qheads;
        const float a = row[qd + g * hdim + i], b = row[qd + g * hdim + i + half];
        const float ka = __fsub_rn(__fmul_rn(a, c), __fmul_rn(b, s));
        const float kb = __fadd_rn(__fmul_rn(b, c), __fmul_rn(a, s));
        const size_t base = pg.row(t, pos, kv_seq_stride, kvd) + (size_t)g * hdim;
        kc[base + i] = f2h(ka);
        kc[base + i + half] = f2h(kb);
        vc[base + i] = f2h(row[qd + kvd + g * hdim + i]);
        vc[base + i + half] = f2h(row[qd + kvd + g * hdim + i + half]);
    }
}

void launch_rope_kv(const float *qkv, int ldqkv, int ntok, int qheads, int kvheads, int hdim,
                    int pos0, int pos_step, int max_pos, const int *ctx_dev, const float *rc,
                    const float *rs, float *q_out, uint16_t *kc, uint16_t *vc,
                    size_t kv_seq_stride, hipStream_t st, KvPages pg) {
    if (ntok <= 0) return;
    const int pairs = (qheads + kvheads) * (hdim / 2);
    SI_LAUNCH(k_rope_kv, dim3(ntok, (pairs + ROPE_T - 1) / ROPE_T), dim3(ROPE_T), 0, st, qkv,
              ldqkv, qheads, kvheads, hdim, pos0, pos_step, max_pos, ctx_dev, rc, rs,
              q_out, kc, vc, kv_seq_stride, pg);
}

constexpr int ATT_MAXPER = 16;  // query heads per KV group (the 16 MFMA columns)

// Weight of a chunk whose running max is m under the head's max mx.  POW2: the
// maxima are in powers of two (the decode kernels of si_decode.hip); otherwise
// natural (k_attn_decode_mfma).  An empty chunk (m = -inf) weighs 0.
template <bool POW2>
__device__ __forceinline__ float part_weight(float m, float mx) {
    return POW2 ? __builtin_amdgcn_exp2f(m - mx) : expf(m - mx);
}

// grid (qheads, nq), block hdim: merge chunks, normalise, quantize to Q8_0
// (tq/td, optional: the Q8_0 also operand-tiled, q8_tiled_byte).
template <bool POW2>
__global__ void k_attn_combine(int qheads, int hdim, int nsplit, const float *__restrict__ ws_m,
                               const float *__restrict__ ws_l, const float *__restrict__ ws_o,
                               float *__restrict__ attn, int8_t *__restrict__ qs,
                               uint16_t *__restrict__ d, int16_t *__restrict__ bsum,
                               int8_t *__restrict__ tq, uint16_t *__restrict__ td) {
    const int h = blockIdx.x, qi = blockIdx.y, jj = threadIdx.x;
    const size_t base = ((size_t)qi * qheads + h) * nsplit;
    // unrolled: the loads of 8 splits are in flight together
    float mx = -INFINITY;
#pragma unroll 8
    for (int s = 0; s < nsplit; ++s) mx = fmaxf(mx, ws_m[base + s]);
    float l = 0.0f, acc = 0.0f;
#pragma unroll 8
    for (int s = 0; s < nsplit; ++s) {
        // (an empty chunk's output may be unwritten)
        const float ms = ws_m[base + s], w = part_weight<POW2>(ms, mx);
        const float os = ws_o[(base + s) * hdim + jj];
        l = fmaf(ws_l[base + s], w, l);
        acc = fmaf(ms == -INFINITY ? 0.0f : os, w, acc);
    }
    // context <= 0 (only possible through ctx_dev): zero output, as
    // attention_kernels.h:95-98 does
    const float y = mx == -INFINITY ? 0.0f : acc * (1.0f / l);
    const size_t off = (size_t)qi * qheads * hdim + (size_t)h * hdim + jj;
    attn[off] = y;
    if (qs) {
        uint16_t dbits;
        int sum;
        const int q = quant_block_lane(y, dbits, sum);
        qs[off] = (int8_t)q;
        if ((jj & 31) == 0) {
            const size_t bi = off / SI_QK;
            d[bi] = dbits;
            if (bsum) bsum[bi] = (int16_t)sum;
        }
        if (tq) {
            const int qd = qheads * hdim;
            const size_t pb = (size_t)(qi >> 5) * (qd / SI_QK) + (h * hdim + jj) / SI_QK;
            tq[q8_tiled_byte(pb, qi & 31, jj & 31)] = (int8_t)q;
            if ((jj & 31) == 0) td[pb * 32 + (qi & 31)] = dbits;
        }
    }
}

// Block-wide max or sum of one value per thread (blockDim.x a multiple of
// 64, at most 1024): wave reduction, then the wave results in wave order.
__device__ __forceinline__ float block_reduce_1024(float v, float *red, bool is_max) {
    // wave reduction, then the 16 wave results in a fixed order
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(v, off, 64);
        v = is_max ? fmaxf(v, o) : v + o;
    }
    const int wave = threadIdx.x >> 6;
    __syncthreads();  // red[] may still be read from the previous reduction
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    float r = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = is_max ? fmaxf(r, red[w]) : r + red[w];
    return r;
}

// k_attn_combine for many partials (>= 32 per head): grid (qheads, nq),
// block P*hdim, P = 1024/hdim.  The max is taken block-wide; thread
// (group, column) merges the partials s = group, group + P, ... and the P
// group sums are added in group order, so the loads of P partials are in
// flight at once instead of one after another.
template <bool POW2>
__global__ __launch_bounds__(1024) void k_attn_combine_wide(
    int qheads, int hdim, int nsplit, const float *__restrict__ ws_m,
    const float *__restrict__ ws_l, const float *__restrict__ ws_o, float *__restrict__ attn,
    int8_t *__restrict__ qs, uint16_t *__restrict__ d, int16_t *__restrict__ bsum,
    int8_t *__restrict__ tq, uint16_t *__restrict__ td) {
    __shared__ float red_o[1024];
    __shared__ float red_l[32];
    __shared__ float red_m[16];
    const int h = blockIdx.x, qi = blockIdx.y, tid = threadIdx.x;
    const int P = blockDim.x / hdim, grp = tid / hdim, jj = tid % hdim;
    const size_t base = ((size_t)qi * qheads + h) * nsplit;
    float mx = -INFINITY;
    for (int s = tid; s < nsplit; s += blockDim.x) mx = fmaxf(mx, ws_m[base + s]);
    mx = block_reduce_1024(mx, red_m, true);
    float l = 0.0f, acc = 0.0f;
#pragma unroll 4
    for (int s = grp; s < nsplit; s += P) {
        // (an empty chunk's output may be unwritten)
        const float ms = ws_m[base + s], w = part_weight<POW2>(ms, mx);
        const float os = ws_o[(base + s) * hdim + jj];
        l = fmaf(ws_l[base + s], w, l);
        acc = fmaf(ms == -INFINITY ? 0.0f : os, w, acc);
    }
    red_o[tid] = acc;
    if (jj == 0) red_l[grp] = l;
    __syncthreads();
    if (tid >= hdim) return;  // no barrier below
    float a = red_o[jj], lt = red_l[0];
    for (int g = 1; g < P; ++g) {
        a += red_o[g * hdim + jj];
        lt += red_l[g];
    }
    const float y = mx == -INFINITY ? 0.0f : a * (1.0f / lt);
    const size_t off = (size_t)qi * qheads * hdim + (size_t)h * hdim + jj;
    attn[off] = y;
    if (qs) {
        uint16_t dbits;
        int sum;
        const int q = quant_block_lane(y, dbits, sum);
        qs[off] = (int8_t)q;
        if ((jj & 31) == 0) {
            const size_t bi = off / SI_QK;
            d[bi] = dbits;
            if (bsum) bsum[bi] = (int16_t)sum;
        }
        if (tq) {
            const int qd = qheads * hdim;
            const size_t pb = (size_t)(qi >> 5) * (qd / SI_QK) + (h * hdim + jj) / SI_QK;
            tq[q8_tiled_byte(pb, qi & 31, jj & 31)] = (int8_t)q;
            if ((jj & 31) == 0) td[pb * 32 + (qi & 31)] = dbits;
        }
    }
}

// Either combine kernel by partial count, the maxima in powers of two or not.
static void combine(int qheads, int hdim, int nq, int nsplit, bool pow2, const AttnParts &pt,
                    float *attn, int8_t *qs, uint16_t *d, int16_t *bsum, hipStream_t st,
                    int8_t *tq = nullptr, uint16_t *td = nullptr) {
#define CALL(KERNEL, BLOCK)                                                                      \
    SI_LAUNCH(KERNEL, dim3(qheads, nq), dim3(BLOCK), 0, st, qheads, hdim, nsplit, pt.m, pt.l,    \
              pt.o, attn, qs, d, bsum, tq, td)
    if (nsplit >= 32) {
        if (pow2) CALL(k_attn_combine_wide<true>, 1024 / hdim * hdim);
        else CALL(k_attn_combine_wide<false>, 1024 / hdim * hdim);
    } else {
        if (pow2) CALL(k_attn_combine<true>, hdim);
        else CALL(k_attn_combine<false>, hdim);
    }
#undef CALL
}

// ===========================================================================
// Matrix-core decode attention.
//
// One workgroup owns (query, KV group, context chunk); its 4 wavefronts take
// every 4th 16-position tile of the chunk.  Per tile a wavefront computes
//     S^T[pos][head] = K[pos][:] . Q[head][:]        (v_mfma_f32_16x16x32_f16)
// with the GQA group's query heads as the 16 MFMA columns (padded), then an
// online-softmax update per head, then
//     O^T[d][head] += V^T[d][pos] . P[pos][head]     (v_mfma_f32_16x16x16_f16)
// K is read straight from HBM as the MFMA A operand (16 B per lane); V rows
// are staged through LDS and read transposed (the MFMA reduction runs over
// positions).  Q and P are fp32 values split into fp16 hi + lo halves
// (x = hi + lo to 22 bits), each product done twice, so the result keeps
// fp32-level accuracy although the matrix cores take fp16.  The 4 wavefronts'
// (max, sum, unnormalised O) are merged in LDS into one partial per
// workgroup; k_attn_combine merges the chunks.
//
// Layouts (16x16 tiles): MFMA output element (i, j) is held by lane
// j + 16*(i/4), register i%4.  The A/B operands give lane l row/column l%16
// and the k-slice (l/16); A and B use the same k-slice per lane, so any
// consistent assignment of reduction indices to slices is exact.
//
// It serves the calls whose results are few (large batches go to the whole-row
// kernel, attn_rows_nsplit): there one Q8_0 scale that falls to the other side of an
// fp16 tie moves the result by more than 5e-5 of it, so the order of its sums
// and its natural-exponent softmax are kept as they are.  In powers of two it
// would take 0.1-0.4 us less of 5-8 at 2-7 queries of 256 positions, 0.1-1.5
// of 5-24 at 4096.
// ===========================================================================
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int MA_TILE = 16;            // positions per wavefront tile
constexpr int MA_SUPER = 4 * MA_TILE;  // positions per workgroup step
constexpr int MA_VPAD = 16;            // halves of LDS row padding (bank spread)

__device__ __forceinline__ void split_hi_lo(float x, _Float16 &hi, _Float16 &lo) {
    hi = (_Float16)x;
    lo = (_Float16)(x - (float)hi);
}

template <int D>
__global__ void __launch_bounds__(256) k_attn_decode_mfma(
    const float *__restrict__ q, int qheads, int kvheads, const uint16_t *__restrict__ kc,
    const uint16_t *__restrict__ vc, size_t kv_seq_stride, const int *__restrict__ ctx_dev,
    int ctx0, int ctx_step, int max_ctx, int chunk, float scale, float *__restrict__ ws_m,
    float *__restrict__ ws_l, float *__restrict__ ws_o, KvPages pg, int kv_row) {
    constexpr int KS = D / 32;  // k-steps of the score MFMA
    constexpr int DT = D / 16;  // d-tiles of the PV MFMA
    constexpr int VROW = D + MA_VPAD;
    __shared__ __attribute__((aligned(16))) _Float16 v_lds[MA_SUPER * VROW];

    const int sp = blockIdx.x, g = blockIdx.y, qi = blockIdx.z;
    const int nsplit = gridDim.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, grp = lane >> 4;
    const int per = qheads / kvheads;
    int ctx = ctx_dev ? ctx_dev[qi] : ctx0 + qi * ctx_step;
    ctx = min(ctx, max_ctx);
    const int p0 = sp * chunk;
    const int p1 = min(ctx, p0 + chunk);
    const int kvd = kv_row;  // elements per cache row (kvheads * D unless a caller
                             // passes one KV group of a wider cache)
    const uint16_t *kbase = kc + (size_t)g * D;  // + pg.row(qi, pos, ...) per row
    const uint16_t *vbase = vc + (size_t)g * D;

    // Q^T as the B operand: lane holds Q[head = col][d = 8*grp + 32*ks + 0..7]
    h8 qh[KS], ql[KS];
    {
        const bool hv = col < per;
        const float *qrow = q + (size_t)qi * qheads * D + (size_t)(g * per + (hv ? col : 0)) * D;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float x = hv ? qrow[32 * ks + 8 * grp + e] : 0.0f;
                _Float16 hi, lo;
                split_hi_lo(x, hi, lo);
                qh[ks][e] = hi;
                ql[ks][e] = lo;
            }
    }
    float m = -INFINITY, lsum = 0.0f;  // running state of head `col`
    f4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = (f4){0.f, 0.f, 0.f, 0.f};

    for (int s0 = p0; s0 < p1; s0 += MA_SUPER) {
        // stage the step's V rows (clamped to valid rows) into LDS
        constexpr int CHUNKS = MA_SUPER * D / 8;  // 16-byte pieces
#pragma unroll
        for (int c = tid; c < CHUNKS; c += 256) {
            const int r = c / (D / 8), e = (c % (D / 8)) * 8;
            const int pos = min(s0 + r, p1 - 1);
            const uint4 v8 = *(const uint4 *)(vbase + pg.row(qi, pos, kv_seq_stride, kvd) + e);
            *(uint4 *)(&v_lds[r * VROW + e]) = v8;
        }
        __syncthreads();
        const int t0 = s0 + MA_TILE * wave;
        if (t0 < p1) {
            // scores: A = K rows (pos = t0 + col), k-slice grp
            const int kpos = min(t0 + col, p1 - 1);
            const uint16_t *krow = kbase + pg.row(qi, kpos, kv_seq_stride, kvd) + 8 * grp;
            f4 sacc = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                const uint4 kraw = *(const uint4 *)(krow + 32 * ks);
                const h8 ka = __builtin_bit_cast(h8, kraw);
                sacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, qh[ks], sacc, 0, 0, 0);
                sacc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka, ql[ks], sacc, 0, 0, 0);
            }
            // lane holds S^T[pos = t0 + 4*grp + r][head = col]
            float s[4];
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int pos = t0 + 4 * grp + r;
                s[r] = pos < p1 ? sacc[r] * scale : -INFINITY;
                mx = fmaxf(mx, s[r]);
            }
            mx = fmaxf(mx, swap16_f(mx));
            mx = fmaxf(mx, swap32_f(mx));
            const float mnew = fmaxf(m, mx);
            const float alpha = expf(m - mnew);  // 0 while m is -inf
            float p[4], ps = 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                p[r] = expf(s[r] - mnew);
                ps += p[r];
            }
            ps += swap16_f(ps);
            ps += swap32_f(ps);
            lsum = lsum * alpha + ps;
            m = mnew;
            h4 ph, pl;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                _Float16 hi, lo;
                split_hi_lo(p[r], hi, lo);
                ph[r] = hi;
                pl[r] = lo;
            }
            // PV: A = V^T[d = 16*dt + col][pos = 4*grp + r] from this wave's LDS rows
            const _Float16 *vw = &v_lds[(MA_TILE * wave + 4 * grp) * VROW + col];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                h4 va;
#pragma unroll
                for (int r = 0; r < 4; ++r) va[r] = vw[r * VROW + 16 * dt];
                f4 acc = o[dt] * alpha;
                acc = __builtin_amdgcn_mfma_f32_16x16x16f16(va, ph, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x16f16(va, pl, acc, 0, 0, 0);
                o[dt] = acc;
            }
        }
        __syncthreads();  // V rows are overwritten by the next step
    }
    // merge the 4 wavefronts' states into the workgroup's partial (split
    // index sp): each wave rescales its sums to the common max, and the
    // scaled outputs are added in wave order through LDS
    __shared__ float mrg_m[4][16], mrg_l[4][16];
    __shared__ float mrg_o[16 * D];
    if (grp == 0) {
        mrg_m[wave][col] = m;
        mrg_l[wave][col] = lsum;
    }
    __syncthreads();
    const float mall = fmaxf(fmaxf(mrg_m[0][col], mrg_m[1][col]), fmaxf(mrg_m[2][col], mrg_m[3][col]));
    const float w = m == -INFINITY ? 0.0f : expf(m - mall);  // a wave with no positions adds 0
    for (int k = 0; k < 4; ++k) {
        if (wave == k)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int idx = col * D + 16 * dt + 4 * grp + r;
                    const float v = o[dt][r] * w;
                    mrg_o[idx] = k == 0 ? v : mrg_o[idx] + v;
                }
        __syncthreads();
    }
    const size_t pbase = ((size_t)qi * qheads + (size_t)g * per) * nsplit + sp;  // head col 0
    if (wave == 0 && grp == 0 && col < per) {
        float l = 0.0f;
        for (int k = 0; k < 4; ++k)
            if (mrg_m[k][col] != -INFINITY) l += mrg_l[k][col] * expf(mrg_m[k][col] - mall);
        ws_m[pbase + (size_t)col * nsplit] = mall;
        ws_l[pbase + (size_t)col * nsplit] = l;
    }
    for (int idx = tid; idx < per * D; idx += 256)
        ws_o[(pbase + (size_t)(idx / D) * nsplit) * D + idx % D] = mrg_o[idx];
}

// ===========================================================================
// Causal prefill attention (flash attention over 32 x 32 tiles).
//
// The query rows of a KV group are its (token, head) pairs, token-major: row
// r is head r % per of token r / per (per = qheads / kvheads).  A wavefront
// computes 32 consecutive rows, so any group size fills its 32 columns (one
// wavefront per head had left one of eight idle at 7 heads).  A workgroup is
// RT * KW wavefronts: RT row tiles that share each K/V tile staged in LDS,
// times KW wavefronts that take every KW-th 32-position tile of the range.
// The KW states of a row tile meet in LDS at the end, so a long range is
// walked by several wavefronts at once, with no partials in memory and no
// merge launch.  Per tile a wavefront computes
//     S^T[pos][row] = K[pos][:] . Q[row][:]          (v_mfma_f32_32x32x16_f16)
// (Q split into fp16 hi + lo halves, each product done twice, for fp32-level
// scores), the causal mask where the tile reaches a row's position, the online
// softmax per row in powers of two (a row's 32 scores sit in one lane and its
// partner lane ^ 32), then
//     O^T[d][row] += V^T[d][pos] . P^T[pos][row]     (v_mfma_f32_32x32x16_f16)
// The running max and sum of a row then live in the lanes that hold its O^T
// column, so the rescale is a per-lane multiply, and rare (below).  P is split
// into fp16 hi + lo halves like Q (an fp16-only P moves outputs by ~1e-3
// relative, enough to break the prefill == sequential decode agreement the
// reference tests).
//
// Bound: the matrix pipe, 2 * (D/16 + D/16) instructions of ~33 cycles per
// tile (1056 at D = 128) against ~115 VALU operations, 16 of them
// exponentials (~620 cycles), which two wavefronts per SIMD overlap in part: a
// tile takes a SIMD about 1600 cycles, a workgroup's first loads and its
// merge another 8 us.  (Issuing the next tile's scores, or the previous
// tile's weighing, among the exponentials within a wavefront changed nothing:
// 92 and 88 us against 87 at 7B x 2048; the second wavefront already fills
// those gaps.  What helped was fewer VALU operations: 87 -> 77 us.)  K and V
// tiles are copied global -> LDS by buffer loads that write LDS (no staging
// registers, no transposition: V^T operands come from the transposing LDS read),
// their 16-byte chunks permuted within each row on the way so that neither the
// score operands (32 rows, one chunk) nor the transposing reads (4 rows, 4
// chunks) meet in a bank.
//
// 32x32 layouts: output (i, j) is held by lane j + 32*((i/4)%2), register
// (i%4) + 4*(i/8); operand lane l supplies row (or column) l%32 and k-slice
// l/32.  A and B use the same k assignment, so any consistent assignment of
// reduction indices to (slice, element) is exact.
// ===========================================================================
typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 pf_h2 __attribute__((ext_vector_type(2)));
typedef float pf_f2 __attribute__((ext_vector_type(2)));
typedef uint32_t pf_u4 __attribute__((ext_vector_type(4)));
typedef pf_u4 pf_u4u __attribute__((aligned(2)));  // at any fp16 address

constexpr int PF_T = 32;      // query rows per wavefront, positions per K/V tile
constexpr int PF_OPAD = 4;    // floats of padding per merged output row

// LDS slot (16-byte unit within the row) of chunk c of tile row r: the 16
// rows a score operand read takes together, and the 4 rows x 4 chunks of a
// transposing read, spread over the 64 banks
template <int D>
__device__ __forceinline__ int pf_k_slot(int r, int c) {
    if (D == 128) return c ^ (r & 15);
    if (D == 64) return c ^ ((r >> 1) & 7);
    if (D == 32) return c ^ ((r >> 2) & 3);
    const int s = c + ((r >> 2) & 3);  // 12 chunks: a rotation
    return s >= D / 8 ? s - D / 8 : s;
}
template <int D>
__device__ __forceinline__ int pf_v_slot(int r, int c) {
    if (D == 128) return c ^ ((r & 3) << 2);
    if (D == 64) return c ^ (((r >> 1) & 1) << 2);
    return c;  // 4 rows already cover the banks
}
// the chunk whose slot is s
template <int D>
__device__ __forceinline__ int pf_k_chunk(int r, int s) {
    if (D != 96) return pf_k_slot<D>(r, s);  // an XOR
    const int c = s - ((r >> 2) & 3);
    return c < 0 ? c + D / 8 : c;
}

// (fmaxf of matrix results would first canonicalise each; a must come from an
// ordinary operation on those results)
__device__ __forceinline__ float max3_f(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// two values as fp16 hi + lo halves (hi rounded to nearest, lo = x - hi by a
// mixed-precision fma; the plain conversion to hi reads both values first)
__device__ __forceinline__ void split_pair(float x0, float x1, pf_h2 &hi, pf_h2 &lo) {
    hi = __builtin_convertvector((pf_f2){x0, x1}, pf_h2);
    float l0, l1;
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l0) : "v"(hi), "v"(x0));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(l1)
        : "v"(hi), "v"(x1));
    lo = __builtin_convertvector((pf_f2){l0, l1}, pf_h2);
}

// at most VM vector-memory operations of this wavefront outstanding, its LDS
// reads complete
template <int VM>
__device__ __forceinline__ void pf_wait() {
    static_assert(VM <= 63, "vmcnt holds 6 bits");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4));
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void pf_barrier() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// ASYNC: kc and vc are 16-byte aligned (and so is every row, a multiple of 64
// bytes).  Otherwise the tiles come through registers, by loads that take any
// address, and are in LDS when copy() returns.
template <int D, int RT, int KW, bool ASYNC>
__global__ void __launch_bounds__(RT * KW * 64) __attribute__((amdgpu_waves_per_eu(2)))
k_attn_prefill(const float *__restrict__ q, int ntok, int qheads, int kvheads, int pos0,
               const uint16_t *__restrict__ kc, const uint16_t *__restrict__ vc, float scale2,
               float *__restrict__ attn, int8_t *__restrict__ qs, uint16_t *__restrict__ qd,
               int16_t *__restrict__ bsum) {
    constexpr int NWV = RT * KW, NT = NWV * 64, KS = D / 16, DT = D / 32, CH = D / 8;
    constexpr int TB = PF_T * D * 2;            // bytes of a K (or V) tile
    constexpr int TI = TB / 1024;               // copy instructions per tile
    constexpr int TIW = (TI + RT - 1) / RT;     // of one wavefront
    constexpr int OROW = D + PF_OPAD;
    // RT > 1: two stage buffers (K tiles, then V tiles) used in turn, one
    // barrier per step.  RT == 1: each wavefront stages its own tiles, K in
    // sb0 and V in sb1, each refilled as soon as it has been read (no
    // barrier).  At the end the wavefronts' outputs: the first half in sb0,
    // the others in sb1.
    constexpr bool DB = RT > 1;
    constexpr int STAGE = DB ? 2 * KW * TB : KW * TB;
    constexpr int HALF_W = (NWV + 1) / 2, MRG = HALF_W * PF_T * OROW * 4;
    __shared__ __attribute__((aligned(16))) uint8_t sb0[STAGE > MRG ? STAGE : MRG];
    __shared__ __attribute__((aligned(16))) uint8_t sb1[STAGE > MRG ? STAGE : MRG];
    __shared__ float mrg_m[NWV][PF_T], mrg_l[NWV][PF_T];
    __shared__ int64_t rowoff[32 * RT];  // output offset of a row, -1 past the last

    const int per = qheads / kvheads, nrows = ntok * per;
    const int units = (nrows + 32 * RT - 1) / (32 * RT);
    // workgroups of one KV group go to the same XCDs (id % 8) where the group
    // count divides 8; the longest ranges first
    const int g = blockIdx.x % kvheads, unit = units - 1 - blockIdx.x / kvheads;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / RT, rt = wave % RT;
    const int t = lane & 31, hh = lane >> 5;
    const int kvd = kvheads * D;
    const int r0 = unit * 32 * RT;  // the workgroup's first row
    const int wr0 = r0 + 32 * rt;   // this wavefront's
    // last cache rows of the workgroup and of this wavefront's tile
    const int last = pos0 + min(r0 + 32 * RT - 1, nrows - 1) / per;
    const int wlast = pos0 + min(wr0 + 31, nrows - 1) / per;
    const int wfirst = pos0 + min(wr0, nrows - 1) / per;  // its lowest causal limit
    const int steps = last / (PF_T * KW) + 1;
    const int myrow = min(wr0 + t, nrows - 1);
    const int prow = pos0 + myrow / per;  // the row's position: it sees cache rows 0..prow

    // this wavefront's copies of a tile: instruction i takes the 16-byte
    // units 64 i .. 64 i + 63 of the tile (LDS order)
    int crow[TIW], ck[TIW], cv[TIW];
#pragma unroll
    for (int i = 0; i < TIW; ++i) {
        const int p = (rt + RT * i) * 64 + lane;
        const int row = p / CH, slot = p % CH;
        crow[i] = row;
        ck[i] = pf_k_chunk<D>(row, slot) * 16;
        cv[i] = pf_v_slot<D>(row, slot) * 16;  // its own inverse
    }
    const auto copy = [&](const uint16_t *base, uint8_t *dst, int step, const int (&col)[TIW]) {
        const int kv0 = min(step * KW + kw, last / PF_T) * PF_T;  // past the range: the last tile
        const uint16_t *src = base + (size_t)kv0 * kvd + g * D;
        // rows past the last one read it again (masked out)
        const auto at = [&](int i) {
            return (uint32_t)(min(crow[i], last - kv0) * (kvd * 2) + col[i]);
        };
        uint8_t *const to = dst + kw * TB + 1024 * rt;
        if constexpr (ASYNC) {
            const __amdgpu_buffer_rsrc_t rs = buf_rsrc(src, 0x7fffffffu);
#pragma unroll
            for (int i = 0; i < TIW; ++i)
                if (TI % RT == 0 || rt + RT * i < TI) lds_copy16(rs, to + 1024 * RT * i, at(i));
        } else {
            pf_u4 x[TIW];
#pragma unroll
            for (int i = 0; i < TIW; ++i)
                if (TI % RT == 0 || rt + RT * i < TI)
                    x[i] = *(const pf_u4u *)((const uint8_t *)src + at(i));
#pragma unroll
            for (int i = 0; i < TIW; ++i)
                if (TI % RT == 0 || rt + RT * i < TI)
                    *(pf_u4 *)(to + 1024 * RT * i + 16 * lane) = x[i];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
    };
    copy(kc, sb0, 0, ck);
    copy(vc, DB ? sb0 + KW * TB : sb1, 0, cv);

    // Q^T as the B operand of the score MFMA: column t, k-slice hh (columns
    // past the last row repeat it and are never stored)
    const size_t qoff = ((size_t)(myrow / per) * qheads + g * per + myrow % per) * D;
    if (kw == 0 && hh == 0) rowoff[32 * rt + t] = wr0 + t < nrows ? (int64_t)qoff : -1;
    h8 qh[KS], ql[KS];
    {
        const float *qrow = q + qoff + 8 * hh;
        float4 a[KS], b[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            a[ks] = *(const float4 *)(qrow + 16 * ks);
            b[ks] = *(const float4 *)(qrow + 16 * ks + 4);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float x[8] = {a[ks].x, a[ks].y, a[ks].z, a[ks].w,
                                b[ks].x, b[ks].y, b[ks].z, b[ks].w};
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                pf_h2 hi, lo;
                split_pair(x[e], x[e + 1], hi, lo);
                qh[ks][e] = hi[0];
                qh[ks][e + 1] = hi[1];
                ql[ks][e] = lo[0];
                ql[ks][e + 1] = lo[1];
            }
        }
    }

    // operand addresses within a stage: K row t, chunk 2 ks + hh; V rows
    // 16 s2 + 8 e + 4 hh + s / 4 (s = lane % 16), columns 32 dt + 16 (lane /
    // 16 % 2) + 4 (s % 4), as the transposing read takes them
    const int s16 = lane & 15;
    int ka[KS], va[DT];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ka[ks] = kw * TB + t * D * 2 + pf_k_slot<D>(t, 2 * ks + hh) * 16;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        va[dt] = kw * TB + (4 * hh + (s16 >> 2)) * D * 2 +
                 pf_v_slot<D>(s16 >> 2, 4 * dt + 2 * ((lane >> 4) & 1) + ((s16 & 3) >> 1)) * 16 +
                 (s16 & 1) * 8;

    float m = -INFINITY, lsum = 0.0f;  // row t's running max; this lane's share of the sum
    f16v o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = (f16v){};

    const auto load_k = [&](const uint8_t *kt, h8 (&a)[KS]) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a[ks] = *(const h8 *)(kt + ka[ks]);
    };
    const auto scores = [&](const h8 (&a)[KS]) {
        // the lo products first: they round at their own small magnitude
        f16v s = (f16v){};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks], ql[ks], s, 0, 0, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks], qh[ks], s, 0, 0, 0);
        return s;
    };
    h8 ph[2], pl[2];  // the tile's weights
    const auto softmax = [&](f16v s, int kv0) {
        if (kv0 + PF_T - 1 > wfirst) {  // wavefront-uniform: the tile reaches a causal limit
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = kv0 + 8 * (r >> 2) + 4 * hh + (r & 3) <= prow ? s[r] : -INFINITY;
        }
        // (a plain operation reads the matrix results first: the compiler
        // puts the wait states they need before it, which it would not
        // before the inline instructions that follow from it)
        float mx = fmaxf(s[0], s[1]);
#pragma unroll
        for (int r = 2; r < 16; r += 2) mx = max3_f(mx, s[r], s[r + 1]);
        mx = fmaxf(mx, swap32_f(mx));
        // The weights are taken against m, a max of the row so far (in powers
        // of two: scale2 * score) that follows the running max only when that
        // has grown by more than 2^8: weights up to 256 lose nothing, and the
        // rescale of the sums, which some row of the 32 would otherwise ask
        // for in most tiles, becomes rare.  A wavefront's first tiles can lie
        // past a row's limit: its state stays (-inf, 0, 0), no NaN.
        const float mnew = fmaxf(m, mx * scale2);
        if (__ballot(mnew > m + 8.0f)) {
            const float alpha = __builtin_amdgcn_exp2f(m - mnew);
            const float a0 = mnew == -INFINITY ? 1.0f : alpha;
            lsum *= a0;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= a0;
            m = mnew;
        }
        const float mref = m == -INFINITY ? 0.0f : m;
        float ps = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[r], scale2, -mref));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(s[r + 1], scale2, -mref));
            ps += p0;
            ps += p1;
            pf_h2 hi, lo;
            split_pair(p0, p1, hi, lo);
            ph[r >> 3][r & 7] = hi[0];
            ph[r >> 3][(r & 7) + 1] = hi[1];
            pl[r >> 3][r & 7] = lo[0];
            pl[r >> 3][(r & 7) + 1] = lo[1];
        }
        lsum += ps;
    };
    const auto weigh = [&](const uint8_t *vt) {
        // k-step s2 covers positions 16*s2 + 8*(e/4) + 4*hh + e%4 (e = element
        // 0..7), the positions of registers 8*s2 + e of the score output
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int s2 = 0; s2 < 2; ++s2) {
                const h4 v0 = __builtin_bit_cast(h4, lds_read_tr16(vt + va[dt] + 16 * s2 * D * 2));
                const h4 v1 =
                    __builtin_bit_cast(h4, lds_read_tr16(vt + va[dt] + (16 * s2 + 8) * D * 2));
                const h8 a = (h8){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, ph[s2], o[dt], 0, 0, 0);
                o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pl[s2], o[dt], 0, 0, 0);
            }
    };
    if constexpr (DB) {
        // one step: the stage is complete and the other buffer free after the
        // barrier; the next stage's copies run during the whole step
        const auto step = [&](uint8_t *cur, uint8_t *nxt, int st) {
            pf_wait<0>();
            pf_barrier();
            if (st + 1 < steps) {
                copy(kc, nxt, st + 1, ck);
                copy(vc, nxt + KW * TB, st + 1, cv);
            }
            const int kv0 = (st * KW + kw) * PF_T;
            if (kv0 <= wlast) {  // wavefront-uniform
                h8 a[KS];
                load_k(cur, a);
                softmax(scores(a), kv0);
                weigh(cur + KW * TB);
            }
        };
        for (int st = 0; st < steps; st += 2) {
            step(sb0, sb1, st);
            if (st + 1 < steps) step(sb1, sb0, st + 1);
        }
    } else {
        for (int st = 0; st < steps; ++st) {
            const int kv0 = (st * KW + kw) * PF_T;
            if (kv0 > wlast) break;  // wavefront-uniform
            const bool more = kv0 + KW * PF_T <= wlast;
            pf_wait<TIW>();  // K is in; V may still be on its way
            h8 a[KS];
            load_k(sb0, a);
            pf_wait<TIW>();  // K has been read
            if (more) copy(kc, sb0, st + 1, ck);
            softmax(scores(a), kv0);
            if (more)
                pf_wait<TIW>();  // V is in; the next K may still be on its way
            else
                pf_wait<0>();
            weigh(sb1);
            pf_wait<TIW>();  // V has been read
            if (more) copy(vc, sb1, st + 1, cv);
        }
    }
    lsum += swap32_f(lsum);
    pf_wait<0>();  // no copy in flight (a wavefront without tiles never waited for its own)
    __syncthreads();  // every wavefront is done with the stage buffers

    // lane (t, hh) holds O[row t][32*dt + 8*(r/4) + 4*hh + r%4] in o[dt][r]
    {
        float *mo = (float *)(wave < HALF_W ? sb0 : sb1) + (wave % HALF_W) * (PF_T * OROW);
        if (hh == 0) {
            mrg_m[wave][t] = m;
            mrg_l[wave][t] = lsum;
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *(f4 *)(mo + t * OROW + 32 * dt + 8 * r4 + 4 * hh) =
                    (f4){o[dt][4 * r4], o[dt][4 * r4 + 1], o[dt][4 * r4 + 2], o[dt][4 * r4 + 3]};
    }
    __syncthreads();
    // a row's factors for its KW states: 2^(m_k - max) / sum, in mrg_m
    if (tid < 32 * RT) {
        const int w0 = tid >> 5, tr = tid & 31;
        float M = -INFINITY, l = 0.0f, f[KW];
#pragma unroll
        for (int k = 0; k < KW; ++k) M = fmaxf(M, mrg_m[k * RT + w0][tr]);
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            f[k] = __builtin_amdgcn_exp2f(mrg_m[k * RT + w0][tr] - M);
            l = fmaf(mrg_l[k * RT + w0][tr], f[k], l);
        }
        const float inv = 1.0f / l;
#pragma unroll
        for (int k = 0; k < KW; ++k) mrg_m[k * RT + w0][tr] = f[k] * inv;
    }
    __syncthreads();
    // 4 consecutive elements of a row per thread: merge the KW states,
    // quantize (8 lanes hold one Q8_0 block, qwen_one_layer.c:272)
    constexpr int EL = 32 * RT * D / 4;
    static_assert(EL % NT == 0, "whole rounds");
#pragma unroll 2
    for (int e = tid; e < EL; e += NT) {
        const int lr = e / (D / 4), dd = 4 * (e % (D / 4)), w0 = lr >> 5, tr = lr & 31;
        float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int w = k * RT + w0;
            const float *mo = (const float *)(w < HALF_W ? sb0 : sb1) + (w % HALF_W) * (PF_T * OROW);
            const f4 v = *(const f4 *)(mo + tr * OROW + dd);
            const float f = mrg_m[w][tr];
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = fmaf(v[i], f, y[i]);
        }
        uint16_t dbits;
        int sum;
        const uint32_t packed = quant_block_oct(y, dbits, sum);  // every lane of the group
        if (rowoff[lr] < 0) continue;  // whole 8-lane groups
        const size_t off = (size_t)rowoff[lr] + dd;
        *(float4 *)(attn + off) = make_float4(y[0], y[1], y[2], y[3]);
        if (qs) {
            *(uint32_t *)(qs + off) = packed;
            if ((tid & 7) == 0) {
                qd[off / SI_QK] = dbits;
                if (bsum) bsum[off / SI_QK] = (int16_t)sum;
            }
        }
    }
}

// Causal prefill of ntok tokens at positions pos0.. of one sequence whose
// cache rows 0..pos0+ntok-1 are in place (RoPE'd K, V).
bool attn_prefill_supported(int qheads, int kvheads, int hdim) {
    return kvheads > 0 && qheads % kvheads == 0 && qheads / kvheads <= 16 &&
           (hdim == 32 || hdim == 64 || hdim == 96 || hdim == 128);
}

// What si_attention_workspace states for a causal prefill: callers size (and
// si_attention and si_attention_static accept or refuse) by it, as when the
// split tiles' states went through memory.  The kernel itself merges in LDS and
// uses none.
size_t attn_prefill_workspace_bytes(int qheads, int hdim, int ntok) {
    return (size_t)ntok * qheads * 2 * (hdim + 2) * sizeof(float);
}

void launch_attn_prefill(const float *q, int ntok, int qheads, int kvheads, int hdim, int pos0,
                         const uint16_t *kc, const uint16_t *vc, float *attn, int8_t *qs,
                         uint16_t *qd, int16_t *bsum, hipStream_t st) {
    if (ntok <= 0) return;
    const int per = qheads / kvheads;
    const float scale2 = softmax_scale2(hdim);
    // Wavefronts per workgroup, by the number of 32-row tiles.  While they are
    // fewer than two per CU each tile gets a workgroup of its own, its range
    // walked four ways; past that two or four tiles share each staged K/V
    // tile, two ways.  Measured (us, kernel alone; RT x KW = 1x4, 2x2, 4x2;
    // before: one wavefront per head and tokens, the range split in memory):
    //   0.5B 512 tokens (224 tiles)          7.9   10.5   13.0   before 17.2
    //   7B 333 after 1500 (292)             32.3   39.0   50.0          71.2
    //   7B 512 (448)                        15.2   17.6   21.7          31.1
    //   7B 700 after 2000 (616)             80.6   70.3   73.9         113
    //   0.5B 2048 (896)                     26.7   31.0   36.6          59.8
    //   0.5B 4000 (1750)                    77.3   72.8   77.8         144
    //   7B 2048 (1792)                      93.7   81.1   76.8         110
    //   12 heads of 128, 5000 (1876)         186    173    157         315
    const long rows = (long)ntok * per;
    const long tiles = (rows + 31) / 32 * kvheads;
    // Caches off a 16-byte boundary, which the copies into LDS do not take:
    // two tiles by two ways throughout, through registers (us a call, aligned |
    // this | the per-query kernels: 0.5B 512 tokens 8.0 | 12.4 | 19.1, 7B 333
    // after 1500 31.9 | 47.9 | 118, 7B 2048 75.8 | 83.5 | 339).
    const bool async = (((uintptr_t)kc | (uintptr_t)vc) & 15) == 0;
    const int rt = !async                              ? 2
                   : tiles < (hdim <= 64 ? 1024 : 512) ? 1
                   : hdim <= 64 || tiles < 1280        ? 2
                                                       : 4;
    const dim3 grid((unsigned)((rows + 32 * rt - 1) / (32 * rt) * kvheads));
#define PF_CALL(DIM, RT, KW, ASYNC)                                                         \
    SI_LAUNCH((k_attn_prefill<DIM, RT, KW, ASYNC>), grid, dim3(RT * KW * 64), 0, st, q, ntok, \
              qheads, kvheads, pos0, kc, vc, scale2, attn, qs, qd, bsum)
#define PF_DIM(DIM)                                \
    if (!async) PF_CALL(DIM, 2, 2, false);         \
    else if (rt == 1) PF_CALL(DIM, 1, 4, true);    \
    else PF_CALL(DIM, 2, 2, true)
    switch (hdim) {
        case 32: PF_DIM(32); break;
        case 64: PF_DIM(64); break;
        case 96:
            if (rt == 4) PF_CALL(96, 4, 2, true);
            else PF_DIM(96);
            break;
        default:
            if (rt == 4) PF_CALL(128, 4, 2, true);
            else PF_DIM(128);
            break;
    }
#undef PF_DIM
#undef PF_CALL
}

// Context chunks per (query, KV group): enough workgroups to cover the chip
// (>= ~512) while every chunk keeps at least one 64-position step.
int attn_nsplit(int kvheads, int nq, int max_ctx) {
    const int base = kvheads * nq;
    int ns = (512 + base - 1) / base;
    // down to one workgroup step per chunk: the many partials this leaves
    // for a single query go to the wide combine kernel (7B, ctx 4096, cold
    // cache, before the in-workgroup merge: 4-step chunks 22.9 us, 1-step
    // 19.9 us)
    const int maxs = (max_ctx + MA_SUPER - 1) / MA_SUPER;
    if (ns > maxs) ns = maxs;
    return ns < 1 ? 1 : ns;
}

size_t attn_workspace_min(int qheads, int hdim, int kvheads, int nq, int max_ctx) {
    const int ns = attn_nsplit(kvheads, nq, max_ctx);  // one partial per workgroup
    return (size_t)nq * qheads * ns * (hdim + 2) * sizeof(float);
}

// Context chunks of the whole-row kernel for si_attention's queries (0: the
// per-group kernel runs: not the shape, or caches below ROWS_CACHE): chunks of
// about four steps, about 512 workgroups in all (two per CU; workgroups past a
// query's context leave at once), no more than 31 (32 take the wide merge:
// 4.4 -> 8-10 us), and partials within 16 MB or the per-group kernel's.
// Measured (us, kernel + merge; per-group kernel -> this, 512 | 1024 workgroups
// aimed at): 48 queries x 200-4096 positions (7B heads) 104.7 + 4.1 -> 51.5 + 4.5
// | 50.9 + 6.9; 64 x 4096 157 + 4.2 -> 94.8 + 4.2 | 98.3 + 4.5; 20 x 1000-4000
// 43.7 + 4.4 -> 19.9 + 4.4 | 24 + 9; 0.5B heads, 64 x 10-4000 35.5 + 4.1 -> 18.2
// + 4.1.
//
// ROWS_CACHE, over the K and V rows of nq contexts of max_ctx: below it the call
// is its two launches by either kernel (us a call, per-group -> this: 0.5B heads
// 8 x 64-1024 12.1 -> 12.4, 16 x 1024, 8.4 MB, 12.3 -> 12.4; 12 heads of 128, 8
// x 1024, 8.4 MB, 12.3 -> 12.6; 7B 8 x 256 12.3 -> 12.5), and its results are
// few, where a scale that falls to the other side of an fp16 tie moves them by
// more than 5e-5: they stay the per-group kernel's.  Above: 12 heads of 128, 10 x
// 1024, 10.5 MB, 13.8 -> 12.4; 0.5B 24 x 1024, 12.6 MB, 13.6 -> 12.4; 7B 24 x 256,
// 12.6 MB, 15.0 -> 11.5.
constexpr size_t ROWS_CACHE = (size_t)10 << 20;
static int attn_rows_nsplit(int qheads, int kvheads, int hdim, int nq, int max_ctx) {
    if (!dec_rows_ok(qheads, kvheads, hdim, nq)) return 0;
    if ((size_t)nq * max_ctx * kvheads * hdim * 4 < ROWS_CACHE) return 0;
    const int rows = 16 * (4 / kvheads);
    const int ns = min((max_ctx + 4 * rows - 1) / (4 * rows), (512 + nq - 1) / nq);
    const size_t each = (size_t)nq * qheads * (hdim + 2) * sizeof(float);
    const int most = max((int)(((size_t)16 << 20) / each), attn_nsplit(kvheads, nq, max_ctx));
    return max(1, min(ns, min(most, 31)));
}

size_t attn_workspace_bytes(int qheads, int hdim, int kvheads, int nq, int max_ctx) {
    const int ns = max(attn_nsplit(kvheads, nq, max_ctx),
                       attn_rows_nsplit(qheads, kvheads, hdim, nq, max_ctx));
    return (size_t)nq * qheads * ns * (hdim + 2) * sizeof(float);
}

bool attn_supported(int qheads, int kvheads, int hdim) {
    return kvheads > 0 && qheads % kvheads == 0 && qheads / kvheads <= ATT_MAXPER &&
           (hdim == 32 || hdim == 64 || hdim == 96 || hdim == 128);
}

void launch_attention(const float *q, int nq, int qheads, int kvheads, int hdim,
                      const uint16_t *kc, const uint16_t *vc, size_t kv_seq_stride,
                      const int *ctx_dev, int ctx0, int ctx_step, int max_ctx, float *attn,
                      int8_t *qs, uint16_t *d, int16_t *bsum, void *workspace, size_t ws_bytes,
                      hipStream_t st, KvPages pg, int kv_row) {
    if (nq <= 0) return;
    if (kv_row <= 0) kv_row = kvheads * hdim;
    const int nr = attn_rows_nsplit(qheads, kvheads, hdim, nq, max_ctx);
    if (nr > 0 && kv_row == kvheads * hdim &&
        ws_bytes >= (size_t)nq * qheads * nr * (hdim + 2) * sizeof(float) &&
        (((uintptr_t)q | (uintptr_t)workspace) & 15) == 0) {
        launch_attn_rows(q, nq, qheads, kvheads, hdim, kc, vc, kv_seq_stride, ctx_dev, ctx0,
                         ctx_step, max_ctx, nr, workspace, st, pg);
        launch_attn_combine(nq, qheads, hdim, nr, workspace, attn, qs, d, bsum, st);
        return;
    }
    const int ns = attn_nsplit(kvheads, nq, max_ctx);
    int chunk = (max_ctx + ns - 1) / ns;
    chunk = (chunk + MA_SUPER - 1) / MA_SUPER * MA_SUPER;
    const AttnParts pt(workspace, (size_t)nq * qheads * ns, hdim);
    const float scale = 1.0f / sqrtf((float)hdim);  // attention_kernels.h:86
    const dim3 grid(ns, kvheads, nq);
#define SI_ATTN_LAUNCH(DIM)                                                                  \
    SI_LAUNCH(k_attn_decode_mfma<DIM>, grid, dim3(256), 0, st, q, qheads, kvheads, kc,       \
              vc, kv_seq_stride, ctx_dev, ctx0, ctx_step, max_ctx, chunk, scale, pt.m,       \
              pt.l, pt.o, pg, kv_row)
    switch (hdim) {
        case 32: SI_ATTN_LAUNCH(32); break;
        case 64: SI_ATTN_LAUNCH(64); break;
        case 96: SI_ATTN_LAUNCH(96); break;
        default: SI_ATTN_LAUNCH(128); break;
    }
#undef SI_ATTN_LAUNCH
    combine(qheads, hdim, nq, ns, false, pt, attn, qs, d, bsum, st);
}

// Merge of the decode kernels' nsplit partials per query and head (m in powers
// of two).
void launch_attn_combine(int nq, int qheads, int hdim, int nsplit, void *workspace,
                         float *attn, int8_t *qs, uint16_t *d, int16_t *bsum, hipStream_t st,
                         int8_t *tq, uint16_t *td) {
    const AttnParts pt(workspace, (size_t)nq * qheads * nsplit, hdim);
    combine(qheads, hdim, nq, nsplit, true, pt, attn, qs, d, bsum, st, tq, td);
}

// ---------------------------------------------------------------------------
// Textbook attention in three stages (attention_standard,
// attention_kernels.h:33-78): the fp32 scores of every (head, position) are
// materialized in a [qheads][context] buffer, normalised in place, then
// weighted into V.  It is the comparison mode of the decode layer; the
// streaming kernels above are the fast path.

// Stage 1, grid (ceil(ctx/64), kvheads), block 256: a workgroup stages the
// K rows of 64 positions of one KV group in LDS (coalesced 16-byte loads,
// each K byte read once per group) and computes the scores of all the
// group's query heads for them: thread (slot, r) owns position t0 + r and
// heads slot, slot + 4, ...  Each dot product is summed in head-dimension
// order with separate multiply and add (the reference's loop under
// -ffp-contract=off), then scaled by 1/sqrt(hdim): the scores match the
// reference's bits.
template <int D>
__global__ __launch_bounds__(256) void k_std_scores(const float *__restrict__ q,
                                                    const uint16_t *__restrict__ kc, int qheads,
                                                    int kvheads, int ctx, float inv,
                                                    float *__restrict__ scores) {
    __shared__ float ks[64][D + 1];  // +1: the dot loop's column reads hit distinct banks
    __shared__ float qsh[ATT_MAXPER][D];
    constexpr int CPR = D / 8;  // 16-byte chunks per K row
    const int g = blockIdx.y, G = qheads / kvheads, t0 = blockIdx.x * 64, tid = threadIdx.x;
    for (int i = tid; i < G * D; i += 256) qsh[i / D][i % D] = q[(size_t)g * G * D + i];
    for (int i = tid; i < 64 * CPR; i += 256) {
        const int r = i / CPR, c = i % CPR;
        const int t = min(t0 + r, ctx - 1);  // rows past the context are loaded, never used
        const uint4 u = *(const uint4 *)(kc + ((size_t)t * kvheads + g) * D + c * 8);
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) ks[r][c * 8 + e] = h2f((uint16_t)(w[e >> 1] >> (16 * (e & 1))));
    }
    __syncthreads();
    const int r = tid & 63, slot = tid >> 6, t = t0 + r;
    if (t >= ctx) return;
    for (int j = slot; j < G; j += 4) {
        float dot = 0.0f;
#pragma unroll 16
        for (int d = 0; d < D; ++d) dot = __fadd_rn(dot, __fmul_rn(qsh[j][d], ks[r][d]));
        scores[(size_t)(g * G + j) * ctx + t] = __fmul_rn(dot, inv);
    }
}

// Stage 2, grid qheads, block 1024: max, exp(s - max) written in place with
// their sum, then multiplied by 1/sum (attention_kernels.h:50-62).
__global__ __launch_bounds__(1024) void k_std_softmax(float *__restrict__ scores, int ctx) {
    __shared__ float red[16];
    float *row = scores + (size_t)blockIdx.x * ctx;
    float m = -INFINITY;
    for (int t = threadIdx.x; t < ctx; t += 1024) m = fmaxf(m, row[t]);
    m = block_reduce_1024(m, red, true);
    float sum = 0.0f;
    for (int t = threadIdx.x; t < ctx; t += 1024) {
        const float e = expf(row[t] - m);
        row[t] = e;
        sum += e;
    }
    const float inv = 1.0f / block_reduce_1024(sum, red, false);
    for (int t = threadIdx.x; t < ctx; t += 1024) row[t] *= inv;
}

// Stage 3, 8 * ceil(qheads * hdim/8 / 8) workgroups of 1024 threads: a
// workgroup owns the 8 output columns 8c..8c+7 of one head (one 16-byte V
// load per position).  Workgroups are dealt to the 8 XCDs in turn (linear
// id % 8), so (head, c) pairs are numbered head-major and each XCD takes a
// contiguous range: the column workgroups of a head, and the heads of a KV
// group, then share their V cache lines in one XCD's L2.
// thread i sums p[t] v[t] over t = i, i + 1024, ... (four loads in flight),
// then the 1024 partial sums are added in a fixed order
// (attention_kernels.h:64-77 up to the summation order).  The normalised
// scores stay in place.
__global__ __launch_bounds__(1024) void k_std_pv(const float *__restrict__ scores,
                                                 const uint16_t *__restrict__ vc, int qheads,
                                                 int kvheads, int hdim, int ctx,
                                                 float *__restrict__ out) {
    __shared__ float red[16][8];
    const int cpr = hdim / 8, npair = qheads * cpr, per_xcd = (npair + 7) / 8;
    const int pair = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (pair >= npair) return;  // whole workgroup: no barrier is skipped
    const int h = pair / cpr, c = pair % cpr, g = h / (qheads / kvheads), tid = threadIdx.x;
    const float *p = scores + (size_t)h * ctx;
    const size_t rstride = (size_t)kvheads * hdim / 8;  // uint4 per cache row
    const uint4 *v = (const uint4 *)vc + (size_t)g * (hdim / 8) + c;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto add = [&](const uint4 u, float pt) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 8; ++e)
            acc[e] = __fadd_rn(acc[e], __fmul_rn(pt, h2f((uint16_t)(w[e >> 1] >> (16 * (e & 1))))));
    };
    int t = tid;
    for (; t + 3 * 1024 < ctx; t += 4 * 1024) {
        uint4 u[4];
        float pt[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            u[k] = v[(size_t)(t + k * 1024) * rstride];
            pt[k] = p[t + k * 1024];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) add(u[k], pt[k]);
    }
    for (; t < ctx; t += 1024) add(v[(size_t)t * rstride], p[t]);
    // fixed-order reduction: butterfly within each wavefront, then the 16
    // wavefront sums in wave order
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
    if ((tid & 63) == 0)
#pragma unroll
        for (int e = 0; e < 8; ++e) red[tid >> 6][e] = acc[e];
    __syncthreads();
    if (tid < 8) {
        float r = red[0][tid];
        for (int w = 1; w < 16; ++w) r += red[w][tid];
        out[(size_t)h * hdim + c * 8 + tid] = r;
    }
}

bool attn_standard_supported(int qheads, int kvheads, int hdim) {
    return kvheads >= 1 && qheads % kvheads == 0 && qheads / kvheads <= ATT_MAXPER &&
           (hdim == 32 || hdim == 64 || hdim == 96 || hdim == 128);
}

void launch_attn_standard(const float *q, int qheads, int kvheads, int hdim, const uint16_t *kc,
                          const uint16_t *vc, int ctx, float *out, float *scores,
                          hipStream_t st) {
    const float inv = 1.0f / sqrtf((float)hdim);
    if (ctx > 0) {
        const dim3 grid((ctx + 63) / 64, kvheads);
        switch (hdim) {  // the head dimensions check_shape admits
        case 32: SI_LAUNCH(k_std_scores<32>, grid, dim3(256), 0, st, q, kc, qheads, kvheads, ctx, inv, scores); break;
        case 64: SI_LAUNCH(k_std_scores<64>, grid, dim3(256), 0, st, q, kc, qheads, kvheads, ctx, inv, scores); break;
        case 96: SI_LAUNCH(k_std_scores<96>, grid, dim3(256), 0, st, q, kc, qheads, kvheads, ctx, inv, scores); break;
        default: SI_LAUNCH(k_std_scores<128>, grid, dim3(256), 0, st, q, kc, qheads, kvheads, ctx, inv, scores); break;
        }
        SI_LAUNCH(k_std_softmax, dim3(qheads), dim3(1024), 0, st, scores, ctx);
    }
    // context 0 leaves the output zero (attention_kernels.h:70)
    const int npair = qheads * (hdim / 8);
    SI_LAUNCH(k_std_pv, dim3(8 * ((npair + 7) / 8)), dim3(1024), 0, st, scores, vc,
              qheads, kvheads, hdim, ctx, out);
}

}  // namespace si
