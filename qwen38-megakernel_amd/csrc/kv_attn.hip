// Split-K decode attention launchers, the L2 prefetch, the combine kernels and prefill attention (gfx950).  The
// decode kernel template is in kv_attn_decode.h.
#include "kv_attn_decode.h"

namespace qkv {

// ------------------------------------------------------------------------------------------------ prefetch
// The first `tiles` tiles of every wave slice of an attention launch's work items copied into LDS and dropped: the
// bytes pass through the L2 of the XCD that workgroup x runs on, and the attention launch with the same arguments puts
// work item x on workgroup x -- the same XCD (workgroups go round-robin over the XCDs by index) -- so its first tile
// copies hit that L2 (or the last-level cache) instead of HBM.  No results: issued ahead of the attention, on another
// stream beside independent work (the reference's pf_l2 in attn_proj, qwen38_mk.cu:2600-2621).
// One workgroup per (sequence, layer, kv head, segment): the launch's n_base work items.  (An attention launch of
// T = 5..8 in two 24-row batches has n_items = 2 n_base; batch b of item x is not item n_base + x, and an index past
// n_base names a layer outside the launch.)  Item x's batches run on workgroups of x's XCD (kv_attn_decode.h), as x does
// here.
template <int KB, int VB>
__global__ __launch_bounds__(256) void k_prefetch(AttnArgs a, int tiles) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const StoreLayout & S = a.S;
    const unsigned st_lds = (unsigned) __builtin_amdgcn_readfirstlane((unsigned) (size_t) (__attribute__((address_space(3))) uint8_t *) smem + wv * STAGE_BYTES);
    for (int item = blockIdx.x; item < a.n_base; item += gridDim.x) {
        int si = 0;
        for (int i = 1; i < a.nseq; i++)
            if (item >= a.sd[i].item0) si = i;
        const SeqDesc sd = a.sd[si];
        const int local = item - sd.item0, seg = local % sd.nseg, lg = local / sd.nseg, g = lg % NKV, l = lg / NKV;
        const int c0 = seg * sd.cs, c1 = min(sd.L, c0 + sd.cs), ntiles = (c1 - c0 + ATP - 1) / ATP;
        const SideLayout SK = S.side[a.layer0 + l][0], SV = S.side[a.layer0 + l][1];
        const size_t ring0 = (size_t) (sd.seq * NKV + g) * S.kvrc;
        for (int i = 0; i < tiles; i++) {
            const int tix = wv + AWAVES * i;
            if (tix >= ntiles) break;
            const int p0 = c0 + ATP * tix, nv = min(ATP, sd.L - p0);
            const int phys = sd.pbase >= 0 ? sd.pbase + p0 / S.page : page_of(S, sd.seq, p0);
            const bool ring = S.kvrc > 0 && p0 >= sd.ws;
            const TileSrc t = tile_src<KB, VB>(S, SK, SV, g, p0, phys, ring0, ring);
            if (ring) issue_tile<8, 8>(t, nv, st_lds, lane);
            else issue_tile<KB, VB>(t, nv, st_lds, lane);
            vm_wait<0>(); // (the stage is reused by the next copy)
        }
    }
}

// ------------------------------------------------------------------------------------------------ output epilogue
// the sigmoid output gate (qwen38_mk.cu:4686)
__device__ __forceinline__ float gated(float v, float g) { return v / (1.0f + expf(-g)); }

// One output row y (head h of token row trow, lane l holding dims 4l .. 4l+3) after the merge: the V un-rotation when
// V is stored rotated, the sigmoid output gate (qwen38_mk.cu:4686) when grow is given, the fp32 store, and when q32a
// is given the o_proj activation units of q32_store (qwen38_mk.cu:283-307): block k = lane / 8 of the head's 8 blocks of
// 32 (j = 8 h + k), amax / 127, round half away from zero; unit gi = 8 h + 2 (k / 2) + half, bytes of the even blocks
// in a, odd ones in b.  All 64 lanes of the wave call it.
__device__ __forceinline__ void finish_row(float (&v)[4], bool vrot, const float * grow, float * orow, int8_t * q32a, int8_t * q32b,
                                           uint16_t * q32m, size_t trow, int h) {
    const int lane = lane_id();
    if (vrot) fwht256_w64(v);
    if (grow) {
        const float4 gt = *reinterpret_cast<const float4 *>(grow + 4 * lane);
        v[0] = gated(v[0], gt.x);
        v[1] = gated(v[1], gt.y);
        v[2] = gated(v[2], gt.z);
        v[3] = gated(v[3], gt.w);
    }
    *reinterpret_cast<float4 *>(orow + 4 * lane) = make_float4(v[0], v[1], v[2], v[3]);
    if (q32a) {
        float am = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
        am = fmaxf(am, shfl_xor(am, 1));
        am = fmaxf(am, shfl_xor(am, 2));
        am = fmaxf(am, shfl_xor(am, 4));
        const float d = am / 127.0f;
        int qv[4];
#pragma unroll
        for (int k = 0; k < 4; k++) qv[k] = am == 0.0f ? 0 : (int) roundf(v[k] / d);
        const int k8 = lane >> 3, part = k8 & 1, hh = (lane >> 2) & 1;
        const size_t gi = trow * 192 + 8 * h + 2 * (k8 >> 1) + hh;
        const unsigned packed = (qv[0] & 0xff) | (qv[1] & 0xff) << 8 | (qv[2] & 0xff) << 16 | (unsigned) (qv[3] & 0xff) << 24;
        *reinterpret_cast<unsigned *>((part ? q32b : q32a) + gi * 16 + 4 * (lane & 3)) = packed;
        int sum = qv[0] + qv[1] + qv[2] + qv[3];
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if ((lane & 3) == 0) {
            q32m[gi * 4 + part] = f2h_bits(d);
            q32m[gi * 4 + 2 + part] = (uint16_t) (int16_t) sum;
        }
    }
}

// ------------------------------------------------------------------------------------------------ combine
// The merge of a head's segment partials (attn_combine, qwen38_mk.cu:4617-4700: y = sum_c e_c O_c / sum_c e_c l_c with
// e_c = exp(m_c - M)).  16 slots: slot s takes the segments c = s, s + 16, .., weighted by exp2(m_c - M_s) against its own
// maximum M_s and summed in segment order; slots 4 w .. 4 w + 3 are merged pairwise, ((0, 1), (2, 3)), then the four
// groups in order (fixed orders: no bit depends on scheduling).  In two forms, the same bits before the epilogue:
//   split form  one workgroup per (output row, 64-dim quarter), for launches without rotated V or o_proj units.  A slot is a
//               16-lane group: 4 waves hold the 16 slots.  The gate, elementwise, is applied here.
//   row form    one workgroup of 16 waves per output row, a slot per wave, then the V un-rotation, gate and o_proj units
//               of the whole row (finish_row).
// A combine waits on one round of loads from beyond the writers' L2s, so both forms have 8 loads per lane at most in
// flight at once (the row form with 4 waves of 32 loads: 7.4 against 5.9 us on 96 rows of 105 segments).
// Both run as a kernel of their own after the attention launch (an in-launch merge by extra workgroups that wait for
// a head's segments measured slower: partials then have to be written through to the coherence point shared by the
// XCDs before the waiting workgroup may read them).
// the output row of a combine workgroup: grid x = row r (times quarters), y = NKV sequence + kv head, z = layer, so that no
// division stands before the first loads (a flat index, and the gate's load ahead of the partials', per call: one layer of
// 4,096 positions 9.93 us, now 9.71; eight short sequences 19.5, now 18.7)
struct CombineRow {
    int l, si, g, r;
};
__device__ __forceinline__ CombineRow combine_row(int r) { return CombineRow{(int) blockIdx.z, (int) (blockIdx.y / NKV), (int) (blockIdx.y % NKV), r}; }

constexpr int CSLOTS = 16, CPER = MAX_SEG / CSLOTS; // slots, segments per slot at most

// one slot's share of a row: segments slot, slot + 16, .. of the head whose segment 0 is item head0, dims dim .. dim + 3
struct CombineRaw {
    float2 ml[CPER];
    float4 o[CPER];
};
struct CombineAcc {
    float4 num;
    float den, M;
};
__device__ __forceinline__ CombineRaw combine_load(const float * __restrict__ part, const float2 * __restrict__ ml_, size_t head0, int nseg, int R,
                                                   int r, int slot, int dim) {
    CombineRaw w;
#pragma unroll
    for (int k = 0; k < CPER; k++) {
        const int c = slot + CSLOTS * k;
        if (c < nseg) {
            w.ml[k] = ml_[(head0 + c) * R + r];
            w.o[k] = *reinterpret_cast<const float4 *>(part + ((head0 + c) * R + r) * HD + dim);
        }
    }
    return w;
}
__device__ __forceinline__ CombineAcc combine_slot(const CombineRaw & w, int nseg, int slot) {
    const float2 (&ml)[CPER] = w.ml;
    const float4 (&o)[CPER] = w.o;
    CombineAcc x{make_float4(0.f, 0.f, 0.f, 0.f), 0.f, -INFINITY};
#pragma unroll
    for (int k = 0; k < CPER; k++)
        if (slot + CSLOTS * k < nseg) x.M = fmaxf(x.M, ml[k].x);
#pragma unroll
    for (int k = 0; k < CPER; k++) {
        if (slot + CSLOTS * k < nseg) {
            const float e = ml[k].x == -INFINITY ? 0.f : exp2f(ml[k].x - x.M);
            x.num.x = __builtin_fmaf(e, o[k].x, x.num.x);
            x.num.y = __builtin_fmaf(e, o[k].y, x.num.y);
            x.num.z = __builtin_fmaf(e, o[k].z, x.num.z);
            x.num.w = __builtin_fmaf(e, o[k].w, x.num.w);
            x.den = __builtin_fmaf(e, ml[k].y, x.den);
        }
    }
    return x;
}
// x weighted by e
__device__ __forceinline__ void combine_scale(CombineAcc & x, float e) {
    x.num.x *= e;
    x.num.y *= e;
    x.num.z *= e;
    x.num.w *= e;
    x.den *= e;
}
// the four groups of slots (sums against maximum md.x, denominators md.y) in order, y = O / l; s_num: group k's float4 at
// s_num[stride k]
__device__ __forceinline__ float4 combine_groups(const float4 * s_num, int stride, const float2 (&md)[AWAVES]) {
    float M = md[0].x;
#pragma unroll
    for (int k = 1; k < AWAVES; k++) M = fmaxf(M, md[k].x);
    float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
    float dd = 0.f;
#pragma unroll
    for (int k = 0; k < AWAVES; k++) {
        const float e = md[k].x == -INFINITY ? 0.f : exp2f(md[k].x - M);
        const float4 z = s_num[stride * k];
        y.x = __builtin_fmaf(e, z.x, y.x);
        y.y = __builtin_fmaf(e, z.y, y.y);
        y.z = __builtin_fmaf(e, z.z, y.z);
        y.w = __builtin_fmaf(e, z.w, y.w);
        dd = __builtin_fmaf(e, md[k].y, dd);
    }
    return make_float4(y.x / dd, y.y / dd, y.z / dd, y.w / dd);
}
// one (row, 64-dim quarter dq) of the output from the row's segment partials; part / ml / out / gate as in AttnArgs, nseg
// and item0 those of the row's sequence si.  The gate's load and the output row's index (a division by T) come after the
// partials' loads
__device__ __forceinline__ void combine_split_core(const float * __restrict__ part, const float2 * __restrict__ ml_, float * out, const float * gate,
                                                   int gs, int R, int T, int nseq, int nseg, int item0, const CombineRow & cr, int dq) {
    __shared__ float4 s_num[AWAVES][16];
    __shared__ float2 s_md[AWAVES];
    const int r = cr.r, g = cr.g, si = cr.si, l = cr.l;
    const size_t head0 = (size_t) item0 + (size_t) (l * NKV + g) * nseg;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, sub = lane >> 4, dl = lane & 15;
    const int dim = 64 * dq + 4 * dl;
    const CombineRaw w = combine_load(part, ml_, head0, nseg, R, r, 4 * wv + sub, dim);
    const int h = GQA * g + r / T, t = r % T;
    const size_t orow = ((size_t) (l * nseq + si) * T + t) * NH + h;
    float4 gt = make_float4(0.f, 0.f, 0.f, 0.f);
    if (gate && wv == 0 && sub == 0) gt = *reinterpret_cast<const float4 *>(gate + orow * gs + dim);
    CombineAcc x = combine_slot(w, nseg, 4 * wv + sub);
    // the wave's 4 lane groups (same dims, slots 4 w .. 4 w + 3)
    const float Mw = quad_max(x.M);
    combine_scale(x, x.M == -INFINITY ? 0.f : exp2f(x.M - Mw));
    x.num.x = quad_sum(x.num.x);
    x.num.y = quad_sum(x.num.y);
    x.num.z = quad_sum(x.num.z);
    x.num.w = quad_sum(x.num.w);
    x.den = quad_sum(x.den);
    if (sub == 0) s_num[wv][dl] = x.num;
    if (lane == 0) s_md[wv] = make_float2(Mw, x.den);
    __syncthreads();
    if (wv == 0 && sub == 0) {
        const float2 md[AWAVES] = {s_md[0], s_md[1], s_md[2], s_md[3]};
        float4 y = combine_groups(&s_num[0][dl], 16, md);
        if (gate) y = make_float4(gated(y.x, gt.x), gated(y.y, gt.y), gated(y.z, gt.z), gated(y.w, gt.w));
        *reinterpret_cast<float4 *>(out + orow * HD + dim) = y;
    }
}

__global__ __launch_bounds__(64 * CSLOTS) void k_combine(AttnArgs a) {
    __shared__ float4 s_num[CSLOTS][64];
    __shared__ float2 s_md[CSLOTS];
    const CombineRow cr = combine_row(blockIdx.x);
    const int r = cr.r, g = cr.g, si = cr.si, l = cr.l, T = a.T;
    const int nseg = a.sd[si].nseg;
    const size_t head0 = (size_t) a.sd[si].item0 + (size_t) (l * NKV + g) * nseg;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const CombineAcc x = combine_slot(combine_load(a.part, a.ml, head0, nseg, a.R, r, wv, 4 * lane), nseg, wv);
    s_num[wv][lane] = x.num;
    if (lane == 0) s_md[wv] = make_float2(x.M, x.den);
    __syncthreads();
    if (wv >= AWAVES) return;
    // wave w merges slots 4 w .. 4 w + 3 pairwise
    {
        float2 md[4];
        float M = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            md[k] = s_md[4 * wv + k];
            M = fmaxf(M, md[k].x);
        }
        CombineAcc y[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            y[k] = CombineAcc{s_num[4 * wv + k][lane], md[k].y, md[k].x};
            combine_scale(y[k], md[k].x == -INFINITY ? 0.f : exp2f(md[k].x - M));
        }
        s_num[4 * wv][lane] = make_float4((y[0].num.x + y[1].num.x) + (y[2].num.x + y[3].num.x), (y[0].num.y + y[1].num.y) + (y[2].num.y + y[3].num.y),
                                          (y[0].num.z + y[1].num.z) + (y[2].num.z + y[3].num.z), (y[0].num.w + y[1].num.w) + (y[2].num.w + y[3].num.w));
        if (lane == 0) s_md[4 * wv] = make_float2(M, (y[0].den + y[1].den) + (y[2].den + y[3].den));
    }
    __syncthreads();
    if (wv == 0) {
        const float2 md[AWAVES] = {s_md[0], s_md[4], s_md[8], s_md[12]};
        const float4 y = combine_groups(&s_num[0][lane], 4 * 64, md);
        float v[4] = {y.x, y.y, y.z, y.w};
        const int h = GQA * g + r / T, t = r % T;
        const size_t trow = (size_t) (l * a.nseq + si) * T + t; // the token's row of 24 x 256 outputs
        finish_row(v, (a.vrot >> (a.layer0 + l)) & 1u, a.gate ? a.gate + (trow * NH + h) * a.gs : nullptr, a.out + (trow * NH + h) * HD,
                   a.q32a, a.q32b, a.q32m, trow, h);
    }
}

__global__ __launch_bounds__(256) void k_combine_split(AttnArgs a) {
    const CombineRow cr = combine_row(blockIdx.x >> 2);
    const SeqDesc & sd = a.sd[cr.si];
    combine_split_core(a.part, a.ml, a.out, a.gate, a.gs, a.R, a.T, a.nseq, sd.nseg, sd.item0, cr, blockIdx.x & 3);
}

// the same for one sequence, with every argument a scalar: they arrive preloaded in SGPRs (kernel-argument preloading,
// build flags of this file), so the partials' loads issue without a round trip to the argument segment first
__global__ __launch_bounds__(256) void k_combine_split1(const float * part, const float2 * ml, float * out, int R, int T, int nseg, int item0,
                                                        const float * gate, int gs) {
    combine_split_core(part, ml, out, gate, gs, R, T, 1, nseg, item0, combine_row(blockIdx.x >> 2), blockIdx.x & 3);
}

// launches whose rows need the whole row in one workgroup (V stored rotated, o_proj units) use the row form
static bool host_combine_needs_rows(const AttnArgs & a) {
    const unsigned vrot = (a.vrot >> a.layer0) & ((a.nl >= 32 ? 0u : 1u << a.nl) - 1u);
    return vrot || a.q32a;
}

hipError_t launch_combine(const AttnArgs & a, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    auto grid = [&](int x) { return dim3((unsigned) (x * a.R), (unsigned) (a.nseq * NKV), (unsigned) a.nl); }; // (combine_row)
    if (host_combine_needs_rows(a)) hipExtLaunchKernelGGL(k_combine, grid(1), dim3(64 * CSLOTS), 0, st, ev0, ev1, 0, a);
    else if (a.nseq == 1)
        hipExtLaunchKernelGGL(k_combine_split1, grid(4), dim3(256), 0, st, ev0, ev1, 0, (const float *) a.part, (const float2 *) a.ml, a.out, a.R, a.T,
                              a.sd[0].nseg, a.sd[0].item0, a.gate, a.gs);
    else hipExtLaunchKernelGGL(k_combine_split, grid(4), dim3(256), 0, st, ev0, ev1, 0, a);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------ prefill
// Causal attention of a group of prefill pieces (pk_attn8's exact form, prefill_attn.cuh:698-702; pieces and window
// prefill_host.cu:606-615), over every layer of a run (equal K / V bits):
//   k_prefill_kv       keys and queries as fp16 MFMA operands in scratch buffers (PrefillArgs::kv16, kq16, q16), each once
//   k_prefill_attn     the attention over them: no unpacking in its loop
//   k_prefill_combine  the segments of each row, the output epilogue
// A piece has up to 30 row blocks of 128 per kv head, and unpacking the stored rows is as much work as a row block's
// share of the attention: done inside the attention kernel, it took half of every workgroup's waves (16,384-position
// prompt: 5.07 ms per layer, 4.19 with the keys unpacked once).  A key is read as its packed row by pieces whose window
// starts after it and as its q8 window row by the others, so both forms are kept: the window's for as long as a piece
// of the call can see it.  With both at hand the pieces of a group need not be stored one by one: up to PF_PIECES of them
// share each launch, the longest contexts first, and a CU that finishes one workgroup goes on to the next (one piece per
// launch left 67 us of starts, ends and short launches around 95 us of tiles).
//
// Keys are cut into absolute segments of a piece's seg positions (a function of its bucket).  Within a segment even and
// odd tiles are two online softmaxes, merged in that order; the combine folds the row's segments 0 .. pos / seg in order:
// each output is a function of its position and the store only, whatever the chunking of the prefill.

// 32 values of scale block b (dims 32 b .. 32 b + 31) of one staged row of B bits -> 16 fp16 pairs fp16_rn(d q) in
// pair order (pair i of word w: o[4 w + i]), the same values as the decode operands (kfrag)
template <int B>
__device__ __forceinline__ void dequant_block(const uint8_t * row, uint16_t sc, int b, half2v (&o)[16]) {
    const half2v d2 = as_h2((unsigned) sc * 0x10001u);
    unsigned W[B == 8 ? 8 : 4], H[3] = {0, 0, 0};
#pragma unroll
    for (int i = 0; i < (B == 8 ? 2 : 1); i++) {
        const uint4 x = reinterpret_cast<const uint4 *>(row + (B == 8 ? 32 : 16) * b)[i];
        W[4 * i] = x.x;
        W[4 * i + 1] = x.y;
        W[4 * i + 2] = x.z;
        W[4 * i + 3] = x.w;
    }
    if constexpr (B < 8) {
        constexpr int HB = B - 4;
#pragma unroll
        for (int i = 0; i < HB; i++) H[i] = reinterpret_cast<const unsigned *>(row + 128 + 4 * HB * b)[i];
    }
#pragma unroll
    for (int w = 0; w < 4; w++) {
        unsigned p[4];
        if constexpr (B == 8) q8_pairs(W[2 * w], W[2 * w + 1], p);
        else code_pairs<B>(W[w], hi_dword<B - 4>(H, w), hi_part<B - 4>(w), p);
#pragma unroll
        for (int i = 0; i < 4; i++) o[4 * w + i] = pair_operand(p[i], i < 2 ? CodeBias<B>::lo : CodeBias<B>::hi, d2);
    }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __fp16 f16v4 __attribute__((__vector_size__(4 * sizeof(__fp16))));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16 at LDS byte address off: in each group of 16 lanes, lane i receives element i % 4 of the 8-byte
// pieces addressed by lanes i / 4 + 4 j, j = 0..3 (as element j)
__device__ __forceinline__ half4 read_tr16(unsigned off) {
    return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) f16v4 *) (size_t) off));
}

// One fp16 tile (32 positions) of the scratch, KV16_TILE bytes: 1 KiB fragments in the order the attention kernel reads
// them, fragment f, lane l at 1024 f + 16 l:
//   f = ks        (16)  A of S^T = K Q^T, K step ks: position l % 32, dims 16 ks + 8 (l / 32) .. + 7 (pair order)
//   f = 16 + 2 db + s2  A of O^T += V^T P^T: dim 32 db + l % 32 (pair order), positions 16 s2 + 8 a + 4 (l / 32) + i as
//                       element 4 a + i
// Copied to LDS as they are, every fragment read is one conflict-free 16-byte read per lane.
constexpr int PQ_REGION = 5120;   // per wave: K rows 2 KB, V rows 2 KB, scales 1 KB of 8 positions
constexpr int SV_LD = HD + 24;    // V rows of the transposing buffer 560 bytes apart: the 4 rows that one 16-lane group of
                                  // a transposed read addresses start 32 bytes apart in the banks
constexpr int PKV_LDS = 4 * PQ_REGION + ATP * SV_LD * 2;
constexpr int SQ_LD = HD + 8;     // query staging rows (halves)
static_assert(PKV_LDS >= 32 * SQ_LD * 2, "query staging");

// the 8 positions of quarter pw of a tile: one wave's copies (5 instructions) into its region
template <int KB, int VB>
__device__ __forceinline__ void pq_issue(const TileSrc & t, int nq, unsigned lds, int lane) {
    constexpr int KRB = 32 * KB, VRB = 32 * VB; // row bytes
#pragma unroll
    for (int j = 0; j < 2; j++) {
        int o = 1024 * j + 16 * lane;
        if (o >= nq * KRB) o = nq * KRB - 16;
        dma16(t.k + o, lds + 1024 * j);
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
        int o = 1024 * j + 16 * lane;
        if (o >= nq * VRB) o = nq * VRB - 16;
        dma16(t.v + o, lds + 2048 + 1024 * j);
    }
    const int r = min(lane & 7, nq - 1);
    dma16(lane < 8 ? static_cast<const void *>(t.ks + 8 * r) : static_cast<const void *>(t.vs + 8 * r), lds + 4096);
}

// one lane: position lane % 8 of its wave's quarter, scale block lane / 8: K straight into the tile's fragments, V into
// the transposing buffer
template <int KB, int VB>
__device__ __forceinline__ void pq_dequant(const uint8_t * reg, int pw, int lane, uint8_t * tile, _Float16 * sV) {
    const int pl = lane & 7, b = lane >> 3, p = 8 * pw + pl;
    const uint16_t * ksc = reinterpret_cast<const uint16_t *>(reg + 4096);
    half2v o[16];
    dequant_block<KB>(reg + pl * 32 * KB, ksc[pl * 8 + b], b, o);
#pragma unroll
    for (int k = 0; k < 4; k++)
        *reinterpret_cast<uint4 *>(tile + 1024 * (2 * b + (k >> 1)) + 16 * (p + 32 * (k & 1))) =
            make_uint4(as_u(o[4 * k]), as_u(o[4 * k + 1]), as_u(o[4 * k + 2]), as_u(o[4 * k + 3]));
    dequant_block<VB>(reg + 2048 + pl * 32 * VB, ksc[64 + pl * 8 + b], b, o);
    uint4 * vd = reinterpret_cast<uint4 *>(sV + p * SV_LD + 32 * b);
#pragma unroll
    for (int k = 0; k < 4; k++) vd[k] = make_uint4(as_u(o[4 * k]), as_u(o[4 * k + 1]), as_u(o[4 * k + 2]), as_u(o[4 * k + 3]));
}

// 32 query rows (block qb of unit u) as fp16 operands: prep, FWHT for rotated K, * 1/16, each wave 8 rows (independent
// loads, one wait), then into fragments: B of S^T = K Q^T, K step ks, lane l: row l % 32, dims 16 ks + 8 (l / 32) .. + 7
// (pair order) at q16 + Q16_BLOCK (u q_blocks + qb) + 1024 ks + 16 l.  Once per row, not once per key segment, and in
// workgroups of their own beside the tiles': in the attention kernel the rows of a workgroup took 13 us before its first
// tile (24 with the prep), as much as 9 pairs of tiles.  Which rows come here: PrefillArgs::q16.
__device__ __forceinline__ void prefill_queries(const PrefillArgs & a, int u, int l, int g, int qb, int wv, int lane, _Float16 * sq) {
    int pi = 0;
#pragma unroll
    for (int i = 1; i < PF_PIECES; i++)
        if (i < a.np && qb >= a.pc[i].qb0) pi = i;
    const PrefillPiece P = a.pc[pi];
    const float * const q = a.q + ((size_t) l * a.T + P.t0) * NH * a.qs;
    const float * const qnw = a.qnw ? a.qnw + (size_t) l * HD : nullptr;
    const bool krot = (a.krot >> (a.layer + l)) & 1u;
    const int r0 = 32 * (qb - P.qb0);
    float4 xs[8];
#pragma unroll
    for (int v = 0; v < 8; v++) {
        const int r = r0 + 8 * wv + v, t = r / GQA, hh = r - GQA * t;
        xs[v] = r < P.R ? *reinterpret_cast<const float4 *>(q + ((size_t) t * NH + GQA * g + hh) * a.qs + 4 * lane)
                        : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int v = 0; v < 8; v++) {
        const int rl = 8 * wv + v, r = r0 + rl;
        half2v o0 = {(_Float16) 0.f, (_Float16) 0.f}, o1 = o0;
        if (r < P.R) {
            const int t = r / GQA;
            float y[4] = {xs[v].x, xs[v].y, xs[v].z, xs[v].w};
            if (qnw) qk_prep(y, qnw, a.rope + (size_t) (P.n0 + t) * 32);
            if (krot) fwht256_w64(y);
            o0[0] = (_Float16) (y[0] * 0.0625f); // (pair order, as the K fragments)
            o0[1] = (_Float16) (y[2] * 0.0625f);
            o1[0] = (_Float16) (y[1] * 0.0625f);
            o1[1] = (_Float16) (y[3] * 0.0625f);
        }
        *reinterpret_cast<uint2 *>(sq + rl * SQ_LD + 4 * lane) = make_uint2(as_u(o0), as_u(o1));
    }
    __syncthreads();
    uint8_t * const dst = a.q16 + ((size_t) u * a.q_blocks + qb) * Q16_BLOCK;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int ks = 4 * wv + k;
        *reinterpret_cast<uint4 *>(dst + 1024 * ks + 16 * lane) =
            *reinterpret_cast<const uint4 *>(sq + (lane & 31) * SQ_LD + 16 * ks + 8 * (lane >> 5));
    }
}

// Blocks 0 .. q_blocks - 1 of a unit (layer, kv head): its query rows (prefill_queries).  The others: tiles p0 .. p1 - 1
// (main rows) and q0 .. q1 - 1 (window rows), one workgroup of 4 waves per tile, each wave copying 8 positions HBM -> LDS
// and unpacking what it copied.  HBM-bound: 4 workgroups per CU (38 KiB of LDS each) keep copies in flight.
template <int KB, int VB>
__global__ __launch_bounds__(256) void k_prefill_kv(PrefillArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t smem[PKV_LDS];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const StoreLayout & S = a.S;
    const int u = blockIdx.y, l = u / a.ng, g = a.g0 + u % a.ng;
    if ((int) blockIdx.x < a.q_blocks) {
        prefill_queries(a, u, l, g, blockIdx.x, wv, lane, reinterpret_cast<_Float16 *>(smem));
        return;
    }
    const int x = blockIdx.x - a.q_blocks, np = a.p1 - a.p0;
    const bool ring = x >= np;
    const int t = ring ? a.q0 + x - np : a.p0 + x;
    const SideLayout SK = S.side[a.layer + l][0], SV = S.side[a.layer + l][1];
    const int p0t = ATP * t, nv = min(ATP, a.L - p0t);
    const int q0 = min(8 * wv, nv - 1), nq = min(8, nv - q0), p0 = p0t + q0;
    const TileSrc src = tile_src<KB, VB>(S, SK, SV, g, p0, page_of(S, a.seq, p0), (size_t) (a.seq * NKV + g) * S.kvrc, ring);
    const unsigned lds = (unsigned) __builtin_amdgcn_readfirstlane(
        (unsigned) (size_t) (__attribute__((address_space(3))) uint8_t *) smem + wv * PQ_REGION);
    uint8_t * const tile = ring ? a.kq16 + ((size_t) u * a.q_tiles + t % a.q_tiles) * KV16_TILE : a.kv16 + ((size_t) u * a.kv_tiles + t) * KV16_TILE;
    uint8_t * const reg = smem + wv * PQ_REGION;
    _Float16 * const sV = reinterpret_cast<_Float16 *>(smem + 4 * PQ_REGION);
    if (ring) {
        pq_issue<8, 8>(src, nq, lds, lane);
        vm_wait<0>();
        pq_dequant<8, 8>(reg, wv, lane, tile, sV);
    } else {
        pq_issue<KB, VB>(src, nq, lds, lane);
        vm_wait<0>();
        pq_dequant<KB, VB>(reg, wv, lane, tile, sV);
    }
    __syncthreads();
    // V fragments by two transposed reads of 4 positions each: lane q + 4 j of 16-lane group gr addresses position
    // 16 s2 + 4 hf + j (+ 8 for the second read), dims 32 db + 16 (gr & 1) + 4 q .. + 3, and lane i of the group receives
    // dim 32 db + 16 (gr & 1) + i of the 4 positions
    const int hf = lane >> 5;
    const unsigned v_lane = (unsigned) (size_t) (const __attribute__((address_space(3))) _Float16 *) sV +
                            2 * ((4 * hf + ((lane >> 2) & 3)) * SV_LD + 16 * ((lane >> 4) & 1) + 4 * (lane & 3));
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int f = 4 * wv + k, db = f >> 1, s2 = f & 1;
        const unsigned vo = v_lane + 2 * (16 * s2 * SV_LD + 32 * db);
        const half8 av = __builtin_shufflevector(read_tr16(vo), read_tr16(vo + 2 * 8 * SV_LD), 0, 1, 2, 3, 4, 5, 6, 7);
        *reinterpret_cast<half8 *>(tile + 1024 * (16 + f) + 16 * lane) = av;
    }
}

// Instruction order for an unrolled chain of N LDS fragment reads each feeding one MFMA: the first D reads, then one
// MFMA and the next read in turn, then the last D MFMAs (scheduling groups; no effect on the arithmetic).  Left to
// itself the scheduler reads each fragment just before its MFMA into the same registers, so every MFMA of the chain
// waits a whole LDS round trip.
constexpr int PF_AHEAD = 4;
template <int D, int N>
__device__ __forceinline__ void pipeline_reads() {
    __builtin_amdgcn_sched_group_barrier(0x100, D, 0); // DS reads
#pragma unroll
    for (int i = 0; i < N - D; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, D, 0);
}

// the order of a tile's O += P V region: the first half's exponentials, then an MFMA, a fragment read and a few of the
// second half's (later the sum's) VALU instructions in turn
__device__ __forceinline__ void pipeline_pv() {
    __builtin_amdgcn_sched_group_barrier(0x002, 24, 0); // VALU
#pragma unroll
    for (int i = 0; i < 16; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // MFMA
        if (i < 16 - PF_AHEAD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
    }
}

// Workgroup = (128 query rows, layer, kv head, key segment), 8 waves: wave w holds rows 32 (w % 4) .. + 31 and runs the
// segment's tiles of parity w / 4 on v_mfma_f32_32x32x16_f16: S^T = K Q^T, P taken straight from the S^T accumulators,
// O^T += V^T P^T.  The two waves of a SIMD hold the same rows on alternate tiles, so one's softmax runs under the
// other's MFMAs.  A pair of tiles (64 KB) is copied HBM / L2 -> LDS while the pair before it is computed: one barrier per
// pair.  At the end the two parities' states are merged through LDS, each wave finishing half of its rows' dims.
// What bounds it: the matrix cores (2,048 cycles per pair of tiles on a SIMD) and the softmax between its two products.
constexpr int PA_BUF = 2 * KV16_TILE;                     // one pair of tiles
constexpr int SY_LD = HD + 4;                             // output rows (floats) of a single-segment piece
constexpr int PA_ML = PF2_ROWS * SY_LD * 4;               // (m, l) of 8 waves x 32 rows, after the pairs and the output rows
constexpr int PA_LDS = PA_ML + 8 * 32 * 8;
static_assert(PA_ML >= 2 * PA_BUF, "two pairs");
static_assert(PA_LDS >= PF2_ROWS * SQ_LD * 2, "query staging inside the tile buffers");

// QPRE: the query operands come from q16 (prefill_queries); otherwise the workgroup prepares its own rows (PrefillArgs::q16).
// A piece of one segment writes its output rows itself (finish_row) instead of partials for the combine.
template <bool QPRE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_prefill_attn(PrefillArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, c = lane & 31, hf = lane >> 5;
    const int par = wv >> 2, wr = wv & 3;
    int pi = 0;
#pragma unroll
    for (int i = 1; i < PF_PIECES; i++)
        if (i < a.np && (int) blockIdx.x >= a.pc[i].blk0) pi = i;
    const PrefillPiece P = a.pc[pi];
    const int combos = a.nl * a.ng * P.nseg, blk = blockIdx.x - P.blk0;
    // a (layer, kv head, segment)'s row blocks on one XCD, side by side (workgroups are dealt to the 8 XCDs round robin):
    // they read the same tiles at about the same time, and the XCD's L2 serves all but the first
    int rb, cb;
    if (combos % 8 == 0) {
        const int nrb = (P.R + PF2_ROWS - 1) / PF2_ROWS, i = blk >> 3, j = i / nrb;
        cb = (blk & 7) + 8 * j;
        rb = i - j * nrb;
    } else {
        rb = blk / combos;
        cb = blk - rb * combos;
    }
    const int k = cb % P.nseg, u = cb / P.nseg, l = u / a.ng, g = a.g0 + u % a.ng;
    const int r0 = PF2_ROWS * rb, rlast = min(P.R, r0 + PF2_ROWS) - 1;
    const int pmax = P.n0 + rlast / GQA;
    const int c0 = k * P.seg;
    if (c0 > pmax) return;
    const int c1 = min(c0 + P.seg, pmax + 1);
    const int ntiles = (c1 - c0 + ATP - 1) / ATP, nsteps = (ntiles + 1) / 2;
    const unsigned lds0 = (unsigned) (size_t) (__attribute__((address_space(3))) uint8_t *) smem;
    const uint8_t * const main0 = a.kv16 + (size_t) u * a.kv_tiles * KV16_TILE + (size_t) wv * (PA_BUF / 8);
    const uint8_t * const win0 = a.kq16 + (size_t) u * a.q_tiles * KV16_TILE + (size_t) wv * (PA_BUF / 8);
    // wave w copies an eighth of the pair of step s (8 KiB) into buffer s % 2: main rows below the window, its q8 rows from
    // there on (the window starts at an even tile and q_tiles is even: a pair never straddles either).  The pair's second
    // tile may lie past the last one of the segment: in bounds (each unit holds a spare tile), its bytes are not used
    auto issue = [&](int s) {
        const int t = c0 / ATP + 2 * s;
        const uint8_t * const src = ATP * t >= P.ws ? win0 + (size_t) (t % max(a.q_tiles, 1)) * KV16_TILE : main0 + (size_t) t * KV16_TILE;
        const unsigned to = (unsigned) __builtin_amdgcn_readfirstlane(lds0 + (s & 1) * PA_BUF + wv * (PA_BUF / 8));
        dma16s_pieces<8, false>(uniform_ptr(src), 16 * lane, to);
    };
    const bool rows = r0 + 32 * wr < P.R; // the wave has rows at all
    half8 qf[16];
    if constexpr (QPRE) {
        issue(0);
        const uint8_t * const qsrc = a.q16 + ((size_t) u * a.q_blocks + P.qb0 + (rows ? r0 / 32 + wr : 0)) * Q16_BLOCK + 16 * lane;
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[ks] = *reinterpret_cast<const half8 *>(qsrc + 1024 * ks);
        // used here, so that the compiler waits for them here and not in the loop, where its wait would also drain the
        // copies of the next pair of tiles
#pragma unroll
        for (int ks = 0; ks < 16; ks++) asm volatile("" : "+v"(qf[ks]));
    } else {
        // all 8 waves stage 16 rows each (prep, FWHT for rotated K, * 1/16, fp16), then take fragments; loaded 8 rows at a
        // time (independent loads, one wait; all 16 at once: 2-7% slower)
        const float * const q = a.q + ((size_t) l * a.T + P.t0) * NH * a.qs;
        const float * const qnw = a.qnw ? a.qnw + (size_t) l * HD : nullptr;
        const bool krot = (a.krot >> (a.layer + l)) & 1u;
        _Float16 * const sq = reinterpret_cast<_Float16 *>(smem);
        for (int jb = 0; jb < 16; jb += 8) {
            float4 xs[8];
#pragma unroll
            for (int v = 0; v < 8; v++) {
                const int r = r0 + 16 * wv + jb + v, t = r / GQA, hh = r - GQA * t;
                xs[v] = r < P.R ? *reinterpret_cast<const float4 *>(q + ((size_t) t * NH + GQA * g + hh) * a.qs + 4 * lane)
                                : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int v = 0; v < 8; v++) {
                const int rl = 16 * wv + jb + v, r = r0 + rl;
                half2v o0 = {(_Float16) 0.f, (_Float16) 0.f}, o1 = o0;
                if (r < P.R) {
                    const int t = r / GQA;
                    const float4 x = xs[v];
                    float y[4] = {x.x, x.y, x.z, x.w};
                    if (qnw) qk_prep(y, qnw, a.rope + (size_t) (P.n0 + t) * 32);
                    if (krot) fwht256_w64(y);
                    o0[0] = (_Float16) (y[0] * 0.0625f); // (pair order, as the K fragments)
                    o0[1] = (_Float16) (y[2] * 0.0625f);
                    o1[0] = (_Float16) (y[1] * 0.0625f);
                    o1[1] = (_Float16) (y[3] * 0.0625f);
                }
                *reinterpret_cast<uint2 *>(sq + rl * SQ_LD + 4 * lane) = make_uint2(as_u(o0), as_u(o1));
            }
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 16; ks++) qf[ks] = *reinterpret_cast<const half8 *>(sq + (32 * wr + c) * SQ_LD + 16 * ks + 8 * hf);
        __syncthreads(); // every wave holds its fragments: the staging area is free
        issue(0);
    }
    const int row = r0 + 32 * wr + c;
    const int lim = row < P.R ? P.n0 + row / GQA : -1;
    const int lim_min = P.n0 + (r0 + 32 * wr) / GQA;
    float m = -INFINITY, ls = 0.f; // running max (log2 units) and sum
    f32x16 O[8];
#pragma unroll
    for (int db = 0; db < 8; db++)
#pragma unroll
        for (int e = 0; e < 16; e++) O[db][e] = 0.f;
    constexpr float RESCALE_LOG2 = 8.f;
    for (int s = 0; s < nsteps; s++) {
        vm_wait<0>();
        __syncthreads(); // the pair of step s is complete, and every wave is done with the buffer of step s - 1
        if (s + 1 < nsteps) issue(s + 1);
        const int i = 2 * s + par;
        if (i >= ntiles || !rows) continue;
        const uint8_t * const tile = smem + (s & 1) * PA_BUF + par * KV16_TILE + 16 * lane;
        const int p0 = c0 + ATP * i;
        f32x16 sacc;
#pragma unroll
        for (int e = 0; e < 16; e++) sacc[e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < 16; ks++)
            sacc = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8 *>(tile + 1024 * ks), qf[ks], sacc, 0, 0, 0);
        pipeline_reads<PF_AHEAD, 16>();
        // the first V fragments, in flight during the softmax
        half8 va[PF_AHEAD];
#pragma unroll
        for (int j = 0; j < PF_AHEAD; j++) va[j] = *reinterpret_cast<const half8 *>(tile + 1024 * (16 + 2 * j));
        if (p0 + ATP - 1 > lim_min) { // fully visible tiles (wave-uniform) skip the causal mask
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int pos = p0 + 8 * (e >> 2) + 4 * hf + (e & 3);
                sacc[e] = pos <= lim ? sacc[e] : -INFINITY;
            }
        }
        // maxima and sums as four independent chains: a wave's own dependent instructions are what a step waits for
        float mx4[4];
#pragma unroll
        for (int e = 0; e < 4; e++) mx4[e] = fmaxf(fmaxf(sacc[e], sacc[4 + e]), fmaxf(sacc[8 + e], sacc[12 + e]));
        float mx = fmaxf(fmaxf(mx4[0], mx4[1]), fmaxf(mx4[2], mx4[3]));
        mx = fmaxf(mx, shfl_xor(mx, 32)) * LOG2E;
        const float mnew = mx > m + RESCALE_LOG2 ? mx : m;
        const float al = m == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mnew); // (O and l are zero before the first key)
        if (__any(al != 1.f)) {
#pragma unroll
            for (int db = 0; db < 8; db++) O[db] *= al;
        }
        const float sh = mnew == -INFINITY ? 0.f : -mnew; // (no visible key yet: every P is exp2(-inf) = 0)
        m = mnew;
        // P of positions 16 s2 .. (half of the tile) and its share of O += P V: the second half's exponentials run under
        // the first half's MFMAs
        half8 pb[2];
#pragma unroll
        for (int s2 = 0; s2 < 2; s2++) {
#pragma unroll
            for (int e = 8 * s2; e < 8 * s2 + 8; e++) {
                sacc[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[e], LOG2E, sh));
                pb[s2][e - 8 * s2] = (_Float16) sacc[e];
            }
#pragma unroll
            for (int db = 0; db < 8; db++) {
                const half8 v = s2 == 0 && db < PF_AHEAD ? va[db] : *reinterpret_cast<const half8 *>(tile + 1024 * (16 + 2 * db + s2));
                O[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v, pb[s2], O[db], 0, 0, 0);
            }
        }
        float ps4[4];
#pragma unroll
        for (int e = 0; e < 4; e++) ps4[e] = (sacc[e] + sacc[4 + e]) + (sacc[8 + e] + sacc[12 + e]);
        float ps = (ps4[0] + ps4[1]) + (ps4[2] + ps4[3]);
        ps += shfl_xor(ps, 32);
        ls = __builtin_fmaf(ls, al, ps);
        pipeline_pv();
    }
    // ---- the two parities of each row, even tiles first: M = max, O = e0 O0 + e1 O1, l likewise.  Each wave gives the
    // other parity's wave half of its dims (blocks 4 (1 - par) .. + 3) and finishes the other half
    float2 * const s_ml = reinterpret_cast<float2 *>(smem + PA_ML);
    __syncthreads();
    if (hf == 0) s_ml[wv * 32 + c] = make_float2(m, ls);
    // values 4 j .. + 3 of dim block db: dims 32 db + 8 j + 4 hf .. + 3 (V's dims are in pair order)
    auto weights = [&](float & M, float & e0, float & e1) {
        const float2 ml0 = s_ml[wr * 32 + c], ml1 = s_ml[(4 + wr) * 32 + c];
        M = fmaxf(ml0.x, ml1.x);
        e0 = ml0.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml0.x - M);
        e1 = ml1.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml1.x - M);
        return __builtin_fmaf(e1, ml1.y, e0 * ml0.y);
    };
    if (P.nseg == 1) { // the output rows: the odd tiles' sums through LDS, merged there, then whole rows per wave
        float * const sy = reinterpret_cast<float *>(smem);
        float * const mine = sy + (32 * wr + c) * SY_LD + 4 * hf;
        if (par == 1) {
#pragma unroll
            for (int db = 0; db < 8; db++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *reinterpret_cast<float4 *>(mine + 32 * db + 8 * j) =
                        make_float4(O[db][4 * j], O[db][4 * j + 2], O[db][4 * j + 1], O[db][4 * j + 3]);
        }
        __syncthreads();
        if (par == 0) {
            float M, e0, e1;
            const float den = weights(M, e0, e1);
#pragma unroll
            for (int db = 0; db < 8; db++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float4 * const at = reinterpret_cast<float4 *>(mine + 32 * db + 8 * j);
                    const float4 z = *at;
                    *at = make_float4(__builtin_fmaf(e1, z.x, e0 * O[db][4 * j]), __builtin_fmaf(e1, z.y, e0 * O[db][4 * j + 2]),
                                      __builtin_fmaf(e1, z.z, e0 * O[db][4 * j + 1]), __builtin_fmaf(e1, z.w, e0 * O[db][4 * j + 3]));
                }
            if (hf == 0) s_ml[wv * 32 + c].y = den; // (only this lane pair reads its row's entries above)
        }
        __syncthreads();
        for (int rl = wv; rl < min(PF2_ROWS, P.R - r0); rl += 8) {
            const float4 x = *reinterpret_cast<const float4 *>(sy + rl * SY_LD + 4 * lane);
            const float den = s_ml[rl].y;
            float v[4] = {x.x / den, x.y / den, x.z / den, x.w / den};
            const int r = r0 + rl, t = r / GQA, h = GQA * g + r - GQA * t;
            const size_t trow = (size_t) l * a.T + P.t0 + t;
            finish_row(v, (a.vrot >> (a.layer + l)) & 1u, a.gate ? a.gate + (trow * NH + h) * a.gs : nullptr, a.out + (trow * NH + h) * HD, a.q32a,
                       a.q32b, a.q32m, trow, h);
        }
        return;
    }
    float4 * const s_o = reinterpret_cast<float4 *>(smem); // [8 waves][16][64]
#pragma unroll
    for (int d = 0; d < 4; d++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float4 x;
            x.x = par ? O[d][4 * j] : O[4 + d][4 * j];
            x.y = par ? O[d][4 * j + 1] : O[4 + d][4 * j + 1];
            x.z = par ? O[d][4 * j + 2] : O[4 + d][4 * j + 2];
            x.w = par ? O[d][4 * j + 3] : O[4 + d][4 * j + 3];
            s_o[(wv * 16 + 4 * d + j) * 64 + lane] = x;
        }
    __syncthreads();
    if (row < P.R) {
        float M, e0, e1;
        const float den = weights(M, e0, e1);
        const size_t at = (size_t) P.part0 + ((size_t) u * P.nseg + k) * P.R + row;
        if (hf == 0 && par == 0) a.ml[at] = make_float2(M, den);
        float * const dst = a.part + at * HD;
        const float4 * const o = s_o + ((wv ^ 4) * 16) * 64 + lane;
#pragma unroll
        for (int d = 0; d < 4; d++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float4 z = o[(4 * d + j) * 64];
                const float zi[4] = {z.x, z.y, z.z, z.w};
                float y[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float own = par ? O[4 + d][4 * j + i] : O[d][4 * j + i];
                    y[i] = par ? __builtin_fmaf(e1, own, e0 * zi[i]) : __builtin_fmaf(e1, zi[i], e0 * own);
                }
                store_part(dst + 32 * (4 * par + d) + 8 * j + 4 * hf, make_float4(y[0], y[2], y[1], y[3]));
            }
    }
}

// One wave per (layer, kv head, row) of the group's pieces of several segments: the row's segments 0 .. pos / seg folded in segment order
// (M' = max(M, m_k), O' = O e^(M - M') + O_k e^(m_k - M'), l likewise; eight at most, pf_seg), y = O / l, then the output
// epilogue.
__global__ __launch_bounds__(256) void k_prefill_combine(PrefillArgs a) {
    const int wid = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int pi = 0;
#pragma unroll
    for (int i = 1; i < PF_PIECES; i++)
        if (i < a.np && wid >= a.pc[i].row0) pi = i;
    const PrefillPiece P = a.pc[pi];
    const int w = wid - P.row0;
    if (P.nseg == 1 || w >= P.R * a.nl * a.ng) return;
    const int r = w % P.R, u = w / P.R, g = a.g0 + u % a.ng, l = u / a.ng;
    const int t = r / GQA, hh = r - GQA * t, pos = P.n0 + t;
    const int nk = pos / P.seg + 1;
    float M = -INFINITY, den = 0.f;
    float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr int RND = 4; // loaded together
    for (int k0 = 0; k0 < nk; k0 += RND) {
        float2 mls[RND];
        float4 os[RND];
#pragma unroll
        for (int j = 0; j < RND; j++)
            if (k0 + j < nk) {
                const size_t at = (size_t) P.part0 + ((size_t) u * P.nseg + k0 + j) * P.R + r;
                mls[j] = a.ml[at];
                os[j] = *reinterpret_cast<const float4 *>(a.part + at * HD + 4 * lane);
            }
#pragma unroll
        for (int j = 0; j < RND; j++)
            if (k0 + j < nk) {
                const float2 ml = mls[j];
                const float4 o = os[j];
                const float Mn = fmaxf(M, ml.x);
                const float e0 = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - Mn);
                const float e1 = ml.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ml.x - Mn);
                num.x = __builtin_fmaf(num.x, e0, e1 * o.x);
                num.y = __builtin_fmaf(num.y, e0, e1 * o.y);
                num.z = __builtin_fmaf(num.z, e0, e1 * o.z);
                num.w = __builtin_fmaf(num.w, e0, e1 * o.w);
                den = __builtin_fmaf(den, e0, e1 * ml.y);
                M = Mn;
            }
    }
    float v[4] = {num.x / den, num.y / den, num.z / den, num.w / den};
    const int h = GQA * g + hh;
    const size_t trow = (size_t) l * a.T + P.t0 + t;
    finish_row(v, (a.vrot >> (a.layer + l)) & 1u, a.gate ? a.gate + (trow * NH + h) * a.gs : nullptr, a.out + (trow * NH + h) * HD, a.q32a,
               a.q32b, a.q32m, trow, h);
}

// ------------------------------------------------------------------------------------------------ dispatch

template <int NP>
static AttnKernel pick(int kb, int vb) {
#define QKV_VB(K)                                                                                                      \
    switch (vb) {                                                                                                      \
    case 4: return k_attn<NP, K, 4>;                                                                                   \
    case 5: return k_attn<NP, K, 5>;                                                                                   \
    case 6: return k_attn<NP, K, 6>;                                                                                   \
    case 7: return k_attn<NP, K, 7>;                                                                                   \
    case 8: return k_attn<NP, K, 8>;                                                                                   \
    default: return nullptr;                                                                                           \
    }
    switch (kb) {
    case 4: QKV_VB(4)
    case 5: QKV_VB(5)
    case 6: QKV_VB(6)
    case 7: QKV_VB(7)
    case 8: QKV_VB(8)
    default: return nullptr;
    }
#undef QKV_VB
}

template <int KB, int VB>
static AttnKernel small_or_null() {
    if constexpr (KB + VB <= 11) return k_attn<1, KB, VB, true>;
    else return nullptr;
}

static AttnKernel pick_small(int kb, int vb) {
#define QKV_VB(K)                                                                                                      \
    switch (vb) {                                                                                                      \
    case 4: return small_or_null<K, 4>();                                                                              \
    case 5: return small_or_null<K, 5>();                                                                              \
    case 6: return small_or_null<K, 6>();                                                                              \
    case 7: return small_or_null<K, 7>();                                                                              \
    default: return nullptr;                                                                                           \
    }
    switch (kb) {
    case 4: QKV_VB(4)
    case 5: QKV_VB(5)
    case 6: QKV_VB(6)
    case 7: QKV_VB(7)
    default: return nullptr;
    }
#undef QKV_VB
}

// CUs of the current device (cached per thread and device)
static int device_cus() {
    static thread_local int dev_cached = -1, cus = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (dev != dev_cached) {
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
        dev_cached = dev;
    }
    return cus;
}

hipError_t launch_attn(const AttnArgs & a, int kb, int vb, int max_blocks, int occ, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    AttnKernel k = nullptr;
    const int np = a.RP / 8;
    // three workgroups per CU (small stages) when one 8-row group of a packed format of at most 11 KiB per tile has
    // more work items than two per CU hold (occ 0), or always (occ 3); occ 2 keeps two
    // (the fused append runs in two-per-CU kernels only)
    const bool small = !a.kin && np == 1 && kb + vb <= 11 && (occ == 3 || (occ == 0 && a.n_items > 2 * device_cus()));
    if (a.kin) k = pick_fused(np, a.wide, kb, vb);
    else if (small) k = pick_small(kb, vb);
    else if (np == 1) k = pick<1>(kb, vb);
    else if (np == 2) k = pick<2>(kb, vb);
    else if (np == 3) k = a.wide ? verify_of<false>(kb, vb) : pick<3>(kb, vb);
    if (!k) return hipErrorInvalidValue;
    static thread_local const void * configured[256];
    static thread_local int n_configured = 0;
    bool done = false;
    for (int i = 0; i < n_configured; i++) done |= configured[i] == (const void *) k;
    const int lds = a.wide ? 2 * (ATTN_LDS + a.RP * HD * 2) : (small ? AWAVES * (1024 * (kb + vb) + 1024) : ATTN_LDS) + a.RP * HD * 2;
    if (!done) {
        const hipError_t e = hipFuncSetAttribute((const void *) k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        if (n_configured < 256) configured[n_configured++] = (const void *) k;
    }
    int blocks = a.n_items;
    if (a.wide) blocks = std::min(blocks, device_cus()); // k_verify: persistent, one workgroup per CU
    if (max_blocks > 0 && blocks > max_blocks) blocks = max_blocks;
    hipExtLaunchKernelGGL(k, dim3(blocks), dim3(a.wide ? 512 : 256), lds, st, ev0, ev1, 0, a);
    return hipGetLastError();
}

typedef void (*PrefillKernel)(PrefillArgs);

static PrefillKernel pick_prefill_kv(int kb, int vb) {
#define QKV_VB(K)                                                                                                      \
    switch (vb) {                                                                                                      \
    case 4: return k_prefill_kv<K, 4>;                                                                                 \
    case 5: return k_prefill_kv<K, 5>;                                                                                 \
    case 6: return k_prefill_kv<K, 6>;                                                                                 \
    case 7: return k_prefill_kv<K, 7>;                                                                                 \
    case 8: return k_prefill_kv<K, 8>;                                                                                 \
    default: return nullptr;                                                                                           \
    }
    switch (kb) {
    case 4: QKV_VB(4)
    case 5: QKV_VB(5)
    case 6: QKV_VB(6)
    case 7: QKV_VB(7)
    case 8: QKV_VB(8)
    default: return nullptr;
    }
#undef QKV_VB
}

hipError_t launch_prefill_kv(const PrefillArgs & a, int kb, int vb, hipStream_t st) {
    PrefillKernel kv = pick_prefill_kv(kb, vb);
    if (!kv) return hipErrorInvalidValue;
    const int blocks = a.q_blocks + a.p1 - a.p0 + a.q1 - a.q0;
    if (blocks > 0) hipLaunchKernelGGL(kv, dim3(blocks, a.nl * a.ng), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_prefill(PrefillArgs & a, hipStream_t st) {
    static thread_local bool configured = false;
    if (!configured) {
        for (PrefillKernel f : {k_prefill_attn<false>, k_prefill_attn<true>}) {
            const hipError_t e = hipFuncSetAttribute((const void *) f, hipFuncAttributeMaxDynamicSharedMemorySize, PA_LDS);
            if (e != hipSuccess) return e;
        }
        configured = true;
    }
    const int units = a.nl * a.ng;
    int blocks = 0, rows = 0, part = 0;
    for (int i = 0; i < a.np; i++) {
        PrefillPiece & P = a.pc[i];
        P.blk0 = blocks;
        P.row0 = rows;
        P.part0 = part;
        blocks += (P.R + PF2_ROWS - 1) / PF2_ROWS * units * P.nseg;
        if (P.nseg == 1) continue; // (the attention writes its output)
        rows += P.R * units;
        part += P.R * units * P.nseg;
    }
    hipLaunchKernelGGL(a.q_blocks ? k_prefill_attn<true> : k_prefill_attn<false>, dim3(blocks), dim3(512), PA_LDS, st, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || rows == 0) return e;
    hipLaunchKernelGGL(k_prefill_combine, dim3((rows + 3) / 4), dim3(256), 0, st, a);
    return hipGetLastError();
}

template <int KB, int VB>
static hipError_t prefetch_kb_vb(const AttnArgs & a, int tiles, hipStream_t st) {
    constexpr int lds = ATTN_LDS;
    static thread_local bool configured = false; // (per instantiation, as launch_attn does)
    if (!configured) {
        const hipError_t e = hipFuncSetAttribute((const void *) k_prefetch<KB, VB>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        configured = true;
    }
    hipLaunchKernelGGL((k_prefetch<KB, VB>), dim3(a.n_base), dim3(256), lds, st, a, tiles);
    return hipGetLastError();
}

hipError_t launch_prefetch(const AttnArgs & a, int kb, int vb, int tiles, hipStream_t st) {
#define QKV_VB(K)                                                                                                      \
    switch (vb) {                                                                                                      \
    case 4: return prefetch_kb_vb<K, 4>(a, tiles, st);                                                                 \
    case 5: return prefetch_kb_vb<K, 5>(a, tiles, st);                                                                 \
    case 6: return prefetch_kb_vb<K, 6>(a, tiles, st);                                                                 \
    case 7: return prefetch_kb_vb<K, 7>(a, tiles, st);                                                                 \
    case 8: return prefetch_kb_vb<K, 8>(a, tiles, st);                                                                 \
    default: return hipErrorInvalidValue;                                                                              \
    }
    switch (kb) {
    case 4: QKV_VB(4)
    case 5: QKV_VB(5)
    case 6: QKV_VB(6)
    case 7: QKV_VB(7)
    case 8: QKV_VB(8)
    default: return hipErrorInvalidValue;
    }
#undef QKV_VB
}

} // namespace qkv
