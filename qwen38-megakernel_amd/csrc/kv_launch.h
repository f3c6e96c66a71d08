// Kernel launchers of the KV path (defined in kv_store.hip / kv_attn*.hip), called by the C-ABI host code.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include "kv_layout.h"

namespace qkv {

// one sequence entry of an attention launch
struct SeqDesc {
    int seq;   // store sequence (lane) index
    int L;     // context length after this call's rows: positions 0 .. L-1
    int ws;    // window start: tiles at positions >= ws are read from the q8 ring
    int cs;    // canonical segment length (a function of L's 640-bucket only)
    int nseg;  // segments: ceil(L / cs) <= 128
    int item0; // first work item of this sequence in the launch
    int pbase; // >= 0: the sequence's pages are pbase, pbase + 1, .. (no table lookup); -1: read the page table
    unsigned nseg_m; // magic31(nseg)
};

// ceil(2^31 / d): floor(n / d) = (2 n * magic31(d)) >> 32 exactly for 0 <= n, 1 <= d with n d < 2^31 (div_m)
inline unsigned magic31(int d) { return (unsigned) (((1ull << 31) + (unsigned) d - 1) / (unsigned) d); }

// The scalars a decode workgroup (k_attn) needs before its first tile copy and for its merge, as 52 dwords at offset 0
// of the kernel arguments: the kernel reads them with four scalar loads and one wait, into registers the
// compiler cannot refill from memory later (it would otherwise re-read fields from the argument segment, each re-read
// a round trip under the launch's load, several of them in series before the first copy).
struct AttnHead {
    uint8_t * kvals; // side0[0]: K of slot layer0
    uint16_t * kscs;
    int8_t * kring;
    uint16_t * krsc;
    uint8_t * vvals; // side0[1]: V of slot layer0
    uint16_t * vscs;
    int8_t * vring;
    uint16_t * vrsc;
    const float * q;       // AttnArgs::q, part, ml, S.ptab, qnw, rope
    float * part;
    float2 * ml;
    const int * ptab;
    const float * qnw;
    const float2 * rope;
    int L, ws, cs, nseg, item0, pbase, seq;                                       // sd[0]
    int n_items, n_base, nseq, T, R, layer0, qs, kvrc, page, n_pages, pt_stride; // AttnArgs / S fields of the same names
    unsigned krot;
    unsigned nseg_m, T_m; // magic31(nseg of sd[0]), magic31(T)
    int pad[3];
};
static_assert(sizeof(AttnHead) == 208, "three 16-dword loads and one 4-dword load");

struct AttnArgs {
    AttnHead h;          // the decode kernels' copy of fields below (fill_head); the others read the fields themselves
    SideLayout side0[2]; // K, V layouts of slot layer0 (S.side[layer0])
    StoreLayout S;
    int layer0;          // first slot of the launch
    int nl;              // layers in the launch (all with the same K/V bits)
    int T, R, RP;        // query tokens, query rows per kv head (6 T), rows per batch: 8 (R <= 8), 16 (R <= 16), else 24
    int nseq;
    int n_base;          // (sequence, layer, kv head, segment) work items
    int n_items;         // n_base (wide), else n_base * ceil(R / RP): every item once per row batch (batch-minor)
    int wide;            // R > 24 in one pass (k_verify: persistent 8-wave workgroups, waves 4..7 holding rows 24..47)
    unsigned krot, vrot; // per-slot bit masks: K / V stored rotated
    SeqDesc sd[8];
    const float * q;     // [nl][nseq][T][NH][HD] queries of this launch's layers (fp32, before the 1/16 scale)
    float * out;         // [nl][nseq][T][NH][HD]
    int qs, gs;          // row strides (floats) of q and gate: 256, or 512 for the q_proj layout [.. NH][q 256 | gate 256]
    const float * qnw;   // optional [nl][HD] q-norm weights: q rows get RMSNorm + RoPE (qk_prep) before use
    const float2 * rope; // with qnw: [positions][32] (cos, sin); row t of a sequence of length L is position L - T + t
    const float * gate;  // optional [nl][nseq][T][NH][gs]: out = y / (1 + exp(-gate))
    int8_t * q32a;       // optional o_proj activation units of out: [nl][nseq][T][192][16] int8 (even blocks)
    int8_t * q32b;       // ... (odd blocks)
    uint16_t * q32m;     // ... [nl][nseq][T][192][4]: half scales of the a / b blocks, int sums of the a / b halves
    float * part;        // [item][R][HD] per-segment partial outputs (unnormalised)
    float2 * ml;         // [item][R] per-segment (max in log2 units, sum)
    // fused append (mk_kv_append_attend): the rows of positions L - T .. L - 1 of every sequence, stored inside this
    // launch by the wave whose tiles hold them, before those tiles are copied.  kin / vin [nseq][T][kin_nl][NKV][HD]
    // (fp16 when kin_f16), layer l of the launch at kin_nl index l; nullptr: no append
    const void * kin;
    const void * vin;
    int kin_nl, kin_f16;
};

// AttnHead from the launch's other fields (after they are final)
inline void fill_head(AttnArgs & a) {
    AttnHead & h = a.h;
    h.kvals = a.side0[0].vals;
    h.kscs = a.side0[0].scs;
    h.kring = a.side0[0].ring;
    h.krsc = a.side0[0].rsc;
    h.vvals = a.side0[1].vals;
    h.vscs = a.side0[1].scs;
    h.vring = a.side0[1].ring;
    h.vrsc = a.side0[1].rsc;
    h.q = a.q;
    h.part = a.part;
    h.ml = a.ml;
    h.ptab = a.S.ptab;
    h.qnw = a.qnw;
    h.rope = a.rope;
    const SeqDesc & d = a.sd[0];
    h.L = d.L;
    h.ws = d.ws;
    h.cs = d.cs;
    h.nseg = d.nseg;
    h.item0 = d.item0;
    h.pbase = d.pbase;
    h.seq = d.seq;
    h.n_items = a.n_items;
    h.n_base = a.n_base;
    h.nseq = a.nseq;
    h.T = a.T;
    h.R = a.R;
    h.layer0 = a.layer0;
    h.qs = a.qs;
    h.kvrc = a.S.kvrc;
    h.page = a.S.page;
    h.n_pages = a.S.n_pages;
    h.pt_stride = a.S.pt_stride;
    h.krot = a.krot;
    h.nseg_m = d.nseg_m;
    h.T_m = magic31(a.T);
    h.pad[0] = h.pad[1] = h.pad[2] = 0;
}

// one prefill piece: the rows of a call that share a 640-position bucket (one window start, one segment length)
struct PrefillPiece {
    int n0, R, ws;  // first query position, 6 rows per token, window start: keys from ws on are the window's q8 rows
    int seg, nseg;  // key positions per segment (pf_seg), ceil(L / seg) segments of the piece's context L
    int t0;         // the piece's first token within the group
    int blk0, row0; // first workgroup of the attention, first row of the combine
    int part0;      // first row of part / ml, in rows
    int qb0;        // first 32-row block of q16
};
constexpr int PF_PIECES = 4; // pieces per launch at most
// a group of consecutive prefill pieces over a run of layers with the same K / V bits: query rows r = 6 t + hh (token t of a
// piece, query head 6 g + hh of kv head g).  Unit u = l ng + (g - g0): layer l of the run, kv head g
struct PrefillArgs {
    StoreLayout S;
    int layer, seq;    // first slot of the run
    int nl, g0, ng;    // layers and kv heads (g0 .. g0 + ng - 1) of the launch
    int np;            // pieces, the longest context first in blk0 order
    PrefillPiece pc[PF_PIECES];
    int T;             // tokens of the whole call (a layer's stride in q, out, gate and the units)
    int L;             // stored positions after the group
    int p0, p1, q0, q1; // tiles that k_prefill_kv writes: p0 .. p1 - 1 from the main rows, q0 .. q1 - 1 from the window's
    int kv_tiles, q_tiles; // tiles per unit of kv16 (main rows) and kq16 (window rows, tile t at t % q_tiles)
    unsigned krot, vrot; // per-slot bit masks: K / V stored rotated
    // 32-row blocks of the group's pieces per unit, and [nl ng][q_blocks][Q16_BLOCK] fp16 operands (kv_attn.hip) of the query
    // rows: done once per row beside the tiles' conversion, not by every segment's workgroup.  For groups with several segments per
    // row whose queries get the prep or the FWHT (16,384 positions, rotated K: 3,838 -> 3,780 us; a prepped 433-token chunk at
    // 60,188 over two layers 1,524 -> 1,455), and for launches of few workgroups, which leave the CUs idle that would share the
    // work: PF_FEW_PREP with the prep or the FWHT (one layer, rotated K: 16 tokens after 500 positions 37.2 -> 32.0 us, 640 after
    // 640, 120 workgroups, 60.0 -> 57.3; prepped 49.5 -> 40.6 and 74.5 -> 69.5; 240 workgroups 65.5 -> 66.0), PF_FEW without
    // (128 after 1,072 46.7 -> 45.4; over four layers, 96 workgroups, 54.3 -> 51.8 but 128 alone 24.4 -> 25.3; 640 alone, 120,
    // 36.5 -> 37.7).  0 otherwise: the extra pass over the queries then costs more than it saves (a 1,111-token prompt without
    // either over four layers 285 -> 300)
    int q_blocks;
    uint8_t * q16;
    const float * q;   // [nl][T][NH][qs] from the group's first token
    int qs;
    const float * qnw; // optional q-norm weights [nl][HD] (the Q prep, table rope)
    const float2 * rope;
    float * out;       // [nl][T][NH][HD]
    const float * gate; // optional [nl][T][NH][gs]
    int gs;
    int8_t * q32a;     // optional o_proj units [nl][T][192][16] (a / b), meta [nl][T][192][4]
    int8_t * q32b;
    uint16_t * q32m;
    uint8_t * kv16;    // [nl ng][kv_tiles][KV16_TILE] fp16 operand tiles (kv_attn.hip) of the main rows
    uint8_t * kq16;    // [nl ng][q_tiles][KV16_TILE] of the window rows
    float * part;      // per piece [nl ng][nseg][R][HD] per-segment partial outputs (unnormalised)
    float2 * ml;       // per piece [nl ng][nseg][R] (max in log2 units, sum)
};
constexpr int KV16_TILE = 2 * ATP * HD * 2; // one tile's K and V as fp16
constexpr int Q16_BLOCK = 32 * HD * 2;      // 32 query rows as fp16
// key positions per prefill segment: 1, 2, 4 or 8 segments over the row's 640-bucket end, in multiples of 128 -- the same for
// every row of a bucket (every row's result is a function of its position).  A workgroup is (128 query rows, kv head,
// segment): a full 640-position piece has 240 of them with two segments, one round on 256 CUs, and more segments repeat
// each workgroup's partial stores.  Short chunks far into a context have few row blocks, so more
// segments pay there (60,000 positions, 2 / 4 / 8 segments: 16 tokens 731 / 412 / 252 us, 256 tokens 706 / 474 / 506, 512
// tokens 830 / 862 / 811, 640 tokens 946 / 962 / 1,003), and up to 20,480 positions whole prompts decide (16,384 with
// four segments: 9% slower).  Rows of one segment need neither partials nor the combine, which were over half of a short
// prompt's time (640 tokens 44 / 38 us with two / one): one segment up to 1,280 positions.  Where the line lies is a trade between
// prompts and short chunks, whose few workgroups then walk all keys one after another.  One q8 layer with the line at 640 /
// 1,280 / 1,920 positions: 1,111 tokens 68 / 52 / 52 us, 640 after 640 55 / 52 / 52 (over four layers 183 / 102 / 101), 128 after
// 1,072 36 / 47 / 46; 1,920 tokens 130 / 107 / 87, 640 after 1,280 65 / 64 / 66, 128 after 1,700 45 / 45 / 61.
inline int pf_seg(int L) {
    const int lb = (L + ATT_BUCKET - 1) / ATT_BUCKET * ATT_BUCKET;
    const int n = lb > 64 * ATT_BUCKET ? 8 : lb > 32 * ATT_BUCKET ? 4 : lb > 2 * ATT_BUCKET ? 2 : 1;
    return 128 * ((lb + 128 * n - 1) / (128 * n));
}
constexpr int PF2_ROWS = 128; // query rows per prefill workgroup (32 per wave)
constexpr int PF_FEW_PREP = 128, PF_FEW = 64; // prefill workgroups of a launch: PrefillArgs::q_blocks

// canonical segment length: 128 ceil(Lb / 16384) positions with Lb = L rounded up to a 640 bucket: a multiple of 4 tiles,
// so the 4 waves of a workgroup stream the same number of tiles; at most 128 segments per kv head (one layer's 4 heads
// fit the 2 workgroup slots of each of the 256 CUs in one pass) and the same partition for every row count T whose rows
// share one bucket
inline __host__ __device__ int seg_len(int L) {
    const int lb = (L + ATT_BUCKET - 1) / ATT_BUCKET * ATT_BUCKET;
    return ATP * AWAVES * ((lb + 16383) / 16384);
}
constexpr int MAX_SEG = 128;
constexpr int STAGE_BYTES = 2 * 32 * 256 + 1024; // one 32-position tile, widest format (q8 K and V) + its scales
constexpr int ATTN_LDS = AWAVES * STAGE_BYTES;   // one stage per wave (+ the query rows: RP * 512 bytes)

// ev0 / ev1: optional events recorded at the kernel's own start and end (hipExtLaunchKernelGGL: the dispatch packet's
// timestamps, the same the profiler reads), for the store's kernel timing
// knw (optional): [nl][HD] k-norm weights; K rows then get RMSNorm + RoPE (qk_prep, table rope) before quantization
hipError_t launch_append(const StoreLayout & S, int seq, int layer0, int nl, int pos, int T, const void * k, const void * v, int f16,
                         hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr, const float * knw = nullptr,
                         const float2 * rope = nullptr);
hipError_t launch_ring_refill(const StoreLayout & S, int seq, int nl, int p0, int p1, hipStream_t st);
// occ: workgroups per CU for one 8-row group of packed formats up to 11 KiB per tile: 0 = three when the launch has more
// work items than two per CU hold, else two; 2 = two; 3 = three
hipError_t launch_attn(const AttnArgs & a, int kb, int vb, int max_blocks, int occ, hipStream_t st, hipEvent_t ev0 = nullptr,
                       hipEvent_t ev1 = nullptr);
// the first `tiles` tiles of every wave slice of the attention launch `a` read into the L2 its workgroups will use
hipError_t launch_prefetch(const AttnArgs & a, int kb, int vb, int tiles, hipStream_t st);
hipError_t launch_combine(const AttnArgs & a, hipStream_t st, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
// the tiles p0 .. and q0 .., and the pieces' query rows, as fp16 operands
hipError_t launch_prefill_kv(const PrefillArgs & a, int kb, int vb, hipStream_t st);
// the group's attention and combine (fills blk0 and row0)
hipError_t launch_prefill(PrefillArgs & a, hipStream_t st);

} // namespace qkv
