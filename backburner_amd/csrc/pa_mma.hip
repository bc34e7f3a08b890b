// pa_mma.hip - partial attention for many query rows per KV head (16-token verify, 512-token prefill chunks, and any
// shape with more than 8 rows) over q8_0 / q4_0 / f16 K and V, head dim 128 (and 256 for long contexts above 64 rows),
// on the matrix cores (gfx950).
//
// One workgroup = one KV head x one block of 32*NW query rows x one chunk of consecutive 32-key tiles; NW waves, 32
// rows each. Per tile the workgroup dequantizes V once into LDS as fp16 (d*q rounded once: the quants become fp16
// integers exactly through the 0x64 exponent byte, then one subtract and one multiply), and K too unless the call takes
// the exact block dots (EX below, which keep K's raw quants), double-buffered, with the next tile's raw bytes already in
// flight into registers. Each wave then computes, with v_mfma_f32_32x32x16_f16,
//   S^T (32 keys x 32 rows) = K . Q'^T      (8 MFMAs over the 128 dims; Q' stays in registers for the whole kernel),
// so lane (h, n) holds row n's scores of keys 8j + 4h + i (j, i < 4) - which is exactly the B operand layout of
//   O^T (128 dims x 32 rows) += V^T . P^T    (4 dim blocks x 2 MFMAs; V^T read from LDS by ds_read_b64_tr_b16),
// so the probabilities never leave registers, and every value a lane holds belongs to its own row n: each half row keeps its
// own running max and sum, exchanged with lane n + 32 where the reference max moves and at the end only. At head dim 256 the
// same with twice the MFMAs, K and V read from LDS a few operands ahead.
//
// What bounds it: a wave issues in order, and at two waves per SIMD its own chain of instructions per tile (about 190 vector
// ones with the exact block dots, 90 without, at 4.5 cycles each, and 16 MFMAs of 32 cycles that they mostly wait for) is the
// time, so what counts is the number of issued instructions on that chain and how evenly the two waves of a SIMD share the
// staging. us per call, before and after the chain was shortened (scales of all blocks in one operand, dots converted by a
// subtraction, page cursors of a few scalar additions, no lane exchange per tile, V staged by the older waves): 4,096 rows x 8
// heads x 65,536 q8_0 keys 1,388 / 1,266, 128 rows x 8 heads x 98,304 q8_0 keys 101.3 / 95.1.
//
// Q' is the query as fp16: PA_QMODE_F16 takes fp16(q*scale) (the reference engines' Qs, phone-attn.h:595-599), and f16
// K in PA_QMODE_GGML fp16(q), K's vec_dot type in ggml's CPU flash_attn_ext (the scale then multiplies the score).
// Quantized K in PA_QMODE_GGML takes exact block dots instead (EX below): Q converted to q8_0 per 32-block as ggml does
// (quantize_row_q8_0_ref), K staged as its raw quants, one int8 MFMA per 32-dim block, and ggml's per-block scaling in
// fp32. Online softmax in base 2 with a reference max that moves only when a score exceeds it by more than 2^MM_PMAX (O is rescaled
// rarely); the exact max is tracked beside it and applied at the end. The row sum adds the fp16 probabilities the PV
// MFMAs consume. Output: one split-K slot per workgroup (O unnormalised against the base-2 max, max, sum), folded by
// the merge kernels, or the final (O, m, l) when the call has a single chunk.
//
// Reference roles: pa_attn_big + pa_big_load (pa-metal.mm:379-487: per (row tile, KV head, key chunk) dequantize a
// K/V block into threadgroup memory as half, S = QK^T on the matrix units, online softmax with key masking, O = a O +
// PV, write a slot); ggml's q8_0 query conversion (restated in oracle/pa_oracle.c, orc_attn_ggml).
#include "pa_mma.h"
#include <hip/hip_ext.h>

namespace pa_hip {

// LDS geometry per head dim: K row stride 2 HD + 16 B (EX: the raw quants, HD + 16 B), so that 16 consecutive keys' 16-byte
// reads hit distinct banks; V row stride 2 HD + 64 B, so that the 4 rows x 64 bytes of a half-wave's transposing reads do;
// and for EX the tile's K block scales, at head dim 128 [key][4 blocks] fp16, at 256 [8 blocks][key] fp32. A stage holds 19,200 B
// at head dim 128, 36,352 at 256.
template <int HD> struct MmGeom {
    static constexpr int NBLK = HD / 32;                      // quant blocks per head row
    static constexpr int KST = 2 * HD + 16, KST8 = HD + 16, VST = 2 * HD + 64;
    static constexpr int KT = 32 * KST, VT = 32 * VST, KSC = 32 * NBLK * (HD == 128 ? 2 : 4);
    static constexpr int STAGE = KT + VT + KSC;
};

// The query rows as the fp16 B operand (lane (h2, n) holds row n, dims 16kk + 8h2 + t): f16(q * scale), or f16(q) for
// f16 K in PA_QMODE_GGML (ggml's f16 vec_dot type)
template <int HD>
__device__ __forceinline__ void mm_prep_q(const AttnArgs & a, uint32_t h, uint32_t row, bool rlive, int h2, mm_h8 (&Qf)[HD / 16]) {
    const float * qrow = a.q + ((size_t) h * a.rows + (rlive ? row : 0)) * HD + 8 * h2;
    const uint32_t qmask = rlive ? 0xffffffffu : 0u;
    const float qs = a.qmode == 0 ? 1.0f : a.scale;
    #pragma unroll
    for (int kk = 0; kk < HD / 16; kk++) {
        const pa_f4 x0 = __builtin_bit_cast(pa_f4, __builtin_bit_cast(pa_u4, *(const pa_f4 *) (qrow + 16 * kk)) & qmask);
        const pa_f4 x1 = __builtin_bit_cast(pa_f4, __builtin_bit_cast(pa_u4, *(const pa_f4 *) (qrow + 16 * kk + 4)) & qmask);
        mm_h8 f;
        #pragma unroll
        for (int t = 0; t < 8; t++) f[t] = (_Float16) pa_f32((t < 4 ? x0[t] : x1[t - 4]) * qs);   // f2h(q * scale)
        Qf[kk] = f;
    }
}

// The query rows as the int8 B operand of the exact block dots (EX): lane (h2, n) holds row n's ggml q8_0 quants of
// dims 32b + 16h2 .. +15 (quantize_row_q8_0_ref: d = amax / 127, id = 1 / d, q = roundf(x * id), d stored as fp16),
// and per block b the (hi, lo) fp16 pair whose
// sum is the fp16 block scale times scale * log2 e (dqb[b], hi in the low half): to about 22 bits where that product
// is at least 2^-9; below, lo falls into the fp16 subnormals and the pair keeps an absolute error of at most 2^-25, so
// the block's term dot_b * dk_b * (hi + lo) errs by at most |dot_b| * dk_b * 2^-25 in base-2 units.
// For q4_0 K (unsigned nibbles u = q + 8 in the int8 MFMA) it also gives, per block, the (hi, lo) pair of
// -8 * (sum of the row's block quants) * (hi + lo) in fp32 (dcb[b]): the offset the unsigned nibbles add to each block
// dot, times the row's scale pair; a key's block scale times it is that block's correction of the score.
template <int HD, int FMT>
__device__ __forceinline__ void mm_prep_qi8(const AttnArgs & a, uint32_t h, uint32_t row, bool rlive, int h2, pa_u4 (&Qi)[HD / 32],
                                            uint32_t (&dqb)[HD / 32], uint32_t (&dcb)[HD / 32]) {
    const float * qrow = a.q + ((size_t) h * a.rows + (rlive ? row : 0)) * HD + 16 * h2;
    const uint32_t qmask = rlive ? 0xffffffffu : 0u;
    const float scale = a.scale;
    #pragma unroll
    for (int b = 0; b < HD / 32; b++) {
        #pragma clang fp contract(off)
        pa_f4 x[4];
        #pragma unroll
        for (int j = 0; j < 4; j++) x[j] = __builtin_bit_cast(pa_f4, __builtin_bit_cast(pa_u4, *(const pa_f4 *) (qrow + 32 * b + 4 * j)) & qmask);
        float am = 0.0f;
        #pragma unroll
        for (int j = 0; j < 4; j++) am = fmaxf(am, fmaxf(fmaxf(fabsf(x[j][0]), fabsf(x[j][1])), fmaxf(fabsf(x[j][2]), fabsf(x[j][3]))));
        am = mm_max32(am);                                           // the block's other 16 values: lane ^ 32
        const float d = am / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const float dq = (float) (_Float16) d * (scale * MM_LOG2E);   // the fp16 block scale * scale, base-2 units
        const _Float16 hi = (_Float16) dq, lo = (_Float16) (dq - (float) hi);
        if constexpr (HD == 256) dqb[b] = __builtin_bit_cast(uint32_t, dq * (FMT == 2 ? 0.0625f : 1.0f));
        else dqb[b] = (uint32_t) __builtin_bit_cast(uint16_t, hi) | ((uint32_t) __builtin_bit_cast(uint16_t, lo) << 16);
        uint32_t w[4];
        int qs = 0;
        #pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t v = 0;
            #pragma unroll
            for (int e = 0; e < 4; e++) {
                const int q = (int) roundf(x[j][e] * id);
                qs += q;
                v |= ((uint32_t) q & 0xffu) << (8 * e);
            }
            w[j] = v;
        }
        Qi[b] = (pa_u4){w[0], w[1], w[2], w[3]};
        if constexpr (FMT == 2 && HD == 128) {
            const auto t = __builtin_amdgcn_permlane32_swap((unsigned) qs, (unsigned) qs, false, false);
            const int qsum = (int) t[0] + (int) t[1];                // the block's 32 quants: lanes l and l ^ 32
            const float c = (float) (-8 * qsum) * ((float) hi + (float) lo);
            const _Float16 chi = (_Float16) c, clo = (_Float16) (c - (float) chi);
            dcb[b] = (uint32_t) __builtin_bit_cast(uint16_t, chi) | ((uint32_t) __builtin_bit_cast(uint16_t, clo) << 16);
        }
    }
}

// Row n's result: the sum over both lanes, O rebased from the reference max to the exact one; the final (O, m, l)
// for a single-chunk call, else split-K slot c
template <int HD>
__device__ __forceinline__ void mm_write_out(const AttnArgs & a, const mm_f16 (&O)[HD / 32], float mref, float mx, float lsum,
                                             uint32_t h, uint32_t row, bool rlive, int h2, uint32_t c) {
    const float lt = mm_sum32(lsum);
    const float f = mref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mref - mx);
    if (!rlive) return;
    const bool direct = a.n_chunks == 1 && a.fused;
    float * dst = direct ? a.O + ((size_t) h * a.rows + row) * HD
                         : a.po + (((size_t) h * a.qr + row) * a.slots + a.slot0 + c) * HD;
    #pragma unroll
    for (int db = 0; db < HD / 32; db++)
        #pragma unroll
        for (int j = 0; j < 4; j++) {
            const pa_f4 v = {O[db][4 * j] * f, O[db][4 * j + 1] * f, O[db][4 * j + 2] * f, O[db][4 * j + 3] * f};
            *(pa_f4 *) (dst + 32 * db + 8 * j + 4 * h2) = v;
        }
    if (h2 == 0) {
        if (direct) {
            a.m[(size_t) h * a.rows + row] = mx == -INFINITY ? -INFINITY : mx * PA_LN2;
            a.l[(size_t) h * a.rows + row] = lt * f;
        } else {
            a.pml[((size_t) h * a.qr + row) * a.slots + a.slot0 + c] = make_float2(mx, lt * f);
        }
    }
}

// EX: exact block dots, as ggml computes them (PA_QMODE_GGML over quantized K). K is staged as its raw quants, with the
// tile's fp16 block scales beside it (q8_0: the int8 quants as they are, half the LDS bytes of the fp16 tile; q4_0: the
// nibbles of one block half as unsigned bytes u = q + 8), and Q as ggml's q8_0 int8 quants. Per 32-block b one
// v_mfma_i32_32x32x32_i8 gives the integer dot itself (|dot| < 2^21), converted to fp32 exactly, and one fp16 MFMA the
// scale product dk_b(key) * (hi + lo)(row) (an outer product: A holds every block's dk twice, block b's B
// operand the row's pair at that block's two places and zeros elsewhere). The scores are the fp32 sum over the blocks of dot_b * (scale product), started
// at -mref: ggml's per-block vec_dot arithmetic (vec_dot_q8_0_q8_0 / q4_0_q8_0), with the softmax scale and the base-2
// conversion inside each block's factor instead of the dot of two fp16-rounded operands. For q4_0 the start value also
// takes the offset of the unsigned nibbles, sum_b dk_b * (-8 * qsum_b) * (hi + lo)_b, from one more MFMA per tile.
// Otherwise (PA_QMODE_F16, f16 K) the QK is one fp16 rounding of each operand and each score is scaled and shifted by
// one fma.
// SKIP: a wave whose 32 rows are all past the call's rows only stages (its share of every tile's loads, dequant and LDS
// stores, and the barriers). For calls with one row block narrower than 32 * NW rows. Without SKIP there is no branch
// there: one costs 13-20 % on full row blocks, as it separates the next tile's loads from the QK MFMAs, which the
// compiler otherwise schedules in one basic block.
// NS = 2 (SKIP, 4 waves, at most 64 rows, one row block): waves 0-1 and 2-3 are two streams that hold the same rows, a step
// stages two tiles and stream x computes the tile 2t + x, where with one stream half the waves of the workgroup (and, as wave i
// of every workgroup runs on SIMD i, half the SIMDs) only stage. The streams fold through LDS at the end, so the slots stay one
// per workgroup. us per call with one stream and with two: 64 rows x 8 heads x 98,304 q4_0 keys 78.0 / 65.2, 40 rows x 33,333
// q4_0 keys 36.8 / 34.0, 48 rows x 65,536 q4_0 keys (fp16 operands) 45.6 / 43.6.
template <int HD, int FMT, int NW, bool SKIP, bool EX, int NS = 1>
__global__ __launch_bounds__(64 * NW, 8 / NW) void mma_kernel(const AttnArgs a) {   // 2 waves per SIMD
    static_assert(!EX || FMT != 0, "the exact block dots take quantized K");
    using G = MmGeom<HD>;
    constexpr int NBLK = G::NBLK;
    // tiles whose raw bytes are in flight in registers (head dim 256: one; O and Q take 192 of the 256 registers there, and
    // a tile's matrix work is twice as long)
    constexpr int PF = HD == 128 && NS == 1 ? 2 : 1;
    constexpr int NT = 64 * NW;
    constexpr int UPT = 128 * NBLK / NT;                             // staging units per thread and tile (128 NBLK per tile)
    constexpr int RW = NW / NS;                                      // row waves per stream
    static_assert(NS == 1 || (SKIP && HD == 128), "several streams come with one partly filled row block");
    static_assert(UPT * NT == 128 * NBLK, "NW must be 4 or 8");
    __shared__ __attribute__((aligned(16))) char smem[2 * NS * G::STAGE];

    // ---- which (chunk, KV head, row block): row blocks fastest, so the workgroups that share a chunk's K/V run side
    // by side on one XCD (= blockIdx % 8 in dispatch order, which takes a contiguous item range) and share its L2
    const uint32_t bid = blockIdx.x, xcd = bid % 8, local = bid / 8;
    const uint32_t t8 = (a.n_items + 7) / 8;
    const uint32_t w = xcd * t8 + local;
    if (local >= t8 || w >= a.n_items) return;
    const uint32_t rb = mm_uni(w % a.nrb), h = mm_uni((w / a.nrb) % a.nkv), c = mm_uni(w / (a.nrb * a.nkv));
    const uint32_t T = a.cstart[a.n_pages];                          // 32-key tiles of the call
    const uint32_t t0 = c * a.chunk, ntiles = min(t0 + a.chunk, T) - t0;   // this chunk's tiles [t0, t0 + ntiles)

    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int n = lane & 31, h2 = lane >> 5;
    const int rw = wave % RW, sx = wave / RW;                        // this wave's 32 rows and stream
    const uint32_t row = rb * (32 * RW) + 32 * rw + n;               // this lane's query row (within the KV head)
    const bool rlive = row < a.rows;
    const bool wlive = !SKIP || rb * (32 * RW) + 32 * rw < a.rows;    // uniform: the wave has a live row

    // ---- staging units of this thread: u = tid + NT*i -> tensor u / (64 NBLK) (uniform),
    // key u / (2 NBLK) & 31, block (u >> 1) & (NBLK - 1), half u & 1; rows past the page's end read zeros (masked later)
    using F = MmFmt<FMT>;
    // the tensor of unit i. With one unit per thread waves 0-3 stage V and waves 4-7 K: V costs the dequantization, and the
    // SIMDs' issue favours the older of its two waves (w and w + 4), so the older one takes it
    static_assert(UPT == 1 || NW == NBLK, "a unit's tensor is then its index, known to the compiler");
    auto unit_tensor = [&](int i) { return UPT == 1 ? 1 - wave / NBLK : i; };
    MmRaw<FMT> R0[NS][UPT], R1[NS][UPT];                             // step t's raw bytes in R(t % PF)
    uint32_t vo[UPT], vq[UPT];                                       // a unit's scale and value bytes in its tile
    #pragma unroll
    for (int i = 0; i < UPT; i++) {
        const uint32_t u = tid + NT * i, key = (u / (2 * NBLK)) & 31, blk = (u >> 1) & (NBLK - 1), half = u & 1;
        vo[i] = key * a.rs + blk * F::BB;
        vq[i] = vo[i] + (FMT == 1 ? 2 + 16 * half : FMT == 2 ? 2 : 32 * half);
    }
    // ---- page cursors (scalar): the loads' (bases of the next tile's rows of this head, keys left in the page) and the
    // matrix work's (keys left). Tiles are taken in order, so a tile costs a few scalar additions and the page table, whose
    // scalar loads would also wait for the LDS operations in flight, is read when a page ends only.
    // The first page comes by shift for uniform pages (a.ptl < 32), else by a walk, one scalar load's latency per page.
    uint32_t lpg = 0;
    if (a.ptl < 32u) lpg = min(t0 >> a.ptl, a.n_pages - 1);
    else while (t0 >= a.cstart[lpg + 1]) lpg++;
    lpg = mm_uni(lpg);
    const uint32_t j00 = 32 * (t0 - a.cstart[lpg]);
    // tiles left in the page and the keys of its last one (no subtraction that stops at zero: that is a vector instruction
    // here, and the descriptors built on its result would take a loop over the lanes per load)
    uint32_t lkeys = mm_uni(a.pstart[lpg + 1] - a.pstart[lpg]), ltl = (lkeys - 1) / 32 + 1 - j00 / 32, llast = (lkeys - 1) % 32 + 1;
    const size_t hoff = (size_t) h * a.hb;
    const uint8_t * lk = mm_uni(a.kp[lpg] + hoff + (size_t) j00 * a.rs), * lv = mm_uni(a.vp[lpg] + hoff + (size_t) j00 * a.rs);
    uint32_t cpg = lpg, ctl = ltl, clast = llast;
    const uint32_t rs32 = 32 * a.rs;
    // buffer loads: the tile's first row of this head as the scalar base, its rows up to the page's end as the range (rows
    // past it read zeros and are masked later). Past the chunk's last tile (live false) the same loads go out with an empty
    // range (no memory access, zeros), so that every step issues the same batch and the wait before a tile's dequant
    // covers its own batch only.
    auto load_one = [&](MmRaw<FMT> (&R)[UPT], bool live) {
        if (live && ltl == 0) {
            do { lpg++; lkeys = a.pstart[lpg + 1] - a.pstart[lpg]; } while (lkeys == 0);
            ltl = (lkeys - 1) / 32 + 1;
            llast = (lkeys - 1) % 32 + 1;
            lk = mm_uni(a.kp[lpg] + hoff);
            lv = mm_uni(a.vp[lpg] + hoff);
            __builtin_amdgcn_s_waitcnt(0xc07f);                      // lgkmcnt(0): no scalar load left outstanding
        }
        // the range covers the tile's rows only (at most 32 of rs bytes, rs < 2^26 by the host's check), so a page of
        // any size keeps the 32-bit byte count exact
        const uint32_t nrec = (live ? (ltl == 1 ? llast : 32u) : 0u) * a.rs;
        #pragma unroll
        for (int i = 0; i < UPT; i++) {
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *) (unit_tensor(i) ? lv : lk), (short) 0, (int) nrec, 0x00020000);
            R[i].q[0] = __builtin_bit_cast(pa_u4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, vq[i], 0, 0));
            if constexpr (FMT == 0) R[i].q[1] = __builtin_bit_cast(pa_u4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, vq[i] + 16, 0, 0));
            R[i].d = FMT == 0 ? 0u : __builtin_amdgcn_raw_buffer_load_b16(rsrc, vo[i], 0, 0);
        }
        lk += rs32;
        lv += rs32;
        ltl -= 1;
    };
    auto load_tile = [&](MmRaw<FMT> (&R)[NS][UPT], uint32_t t) {     // step t's tiles NS t .. NS t + NS - 1
        #pragma unroll
        for (int x = 0; x < NS; x++) load_one(R[x], NS * t + x < ntiles);
    };
    auto store_one = [&](const MmRaw<FMT> (&R)[UPT], char * st) {
        #pragma unroll
        for (int i = 0; i < UPT; i++) {
            const int u = tid + NT * i;
            const int tensor = unit_tensor(i), key = (u / (2 * NBLK)) & 31, blk = (u >> 1) & (NBLK - 1), half = u & 1;
            pa_u4 lo, hi;
            if (EX && tensor == 0) {                                 // K: the raw int8 quants (q4_0: this half's
                                                                     // nibbles as unsigned bytes), the block scale beside
                pa_u4 q = R[i].q[0];
                if constexpr (HD == 128) {
                    if (half == 0) *(uint16_t *) (st + G::KT + G::VT + 2 * NBLK * key + 2 * blk) = (uint16_t) R[i].d;
                    if constexpr (FMT == 2) q = (q >> (4 * half)) & 0x0f0f0f0fu;
                } else {
                    if (half == 0) *(float *) (st + G::KT + G::VT + 4 * (32 * blk + key)) = pa_f16_bits_to_f32((uint16_t) R[i].d);
                    if constexpr (FMT == 2) q = ((q << (4 - 4 * half)) & 0xf0f0f0f0u) ^ 0x80808080u;
                }
                *(pa_u4 *) (st + key * G::KST8 + 32 * blk + 16 * half) = q;
                continue;
            }
            mm_dequant<FMT>(R[i], half, lo, hi);
            char * dst = tensor ? st + G::KT + key * G::VST : st + key * G::KST;
            dst += 2 * (32 * blk + 16 * half);
            *(pa_u4 *) dst = lo;
            *(pa_u4 *) (dst + 16) = hi;
        }
    };

    auto store_tile = [&](const MmRaw<FMT> (&R)[NS][UPT], int stage) {
        #pragma unroll
        for (int x = 0; x < NS; x++) store_one(R[x], smem + (stage * NS + x) * G::STAGE);
    };

    // ---- the first two tiles' loads, then the query rows (B operand: lane (h2, n) holds row n, dims 16kk + 8h2 + t)
    load_tile(R0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PF == 2) load_tile(R1, 1);
    __builtin_amdgcn_sched_barrier(0);
    mm_h8 Qf[HD / 16];                                               // !EX: fp16 query operands
    pa_u4 Qi[NBLK];                                                  // EX: int8 query quants per block
    uint32_t dqb[NBLK], dcb[NBLK];                                   // EX: the scale pairs; q4_0: the nibble-offset pairs
    #pragma unroll
    for (int b = 0; b < NBLK; b++) dqb[b] = dcb[b] = 0u;
    if constexpr (EX) mm_prep_qi8<HD, FMT>(a, h, row, rlive, h2, Qi, dqb, dcb);
    else mm_prep_q<HD>(a, h, row, rlive, h2, Qf);
    // EX at head dim 128: the B operands of the scale products. All four products share one A operand, key n's block scales at k = 2b and
    // 2b + 1 (lanes h2 = b / 2, register b % 2), so block b's B operand holds row n's (hi, lo) pair there, zero elsewhere
    // (one operand per block in otherwise zero registers took four permutes, four selects and eleven moves per tile more)
    pa_u2 dqw[4];
    #pragma unroll
    for (int b = 0; b < 4; b++) {
        const uint32_t x = h2 == (b >> 1) ? dqb[b] : 0u;
        dqw[b] = (b & 1) ? (pa_u2){0u, x} : (pa_u2){x, 0u};
    }
    // EX, q4_0: the correction MFMA's B operand has every block's pair at its place, and its terms k = 4, 5 of lanes
    // h2 = 0 are 1.0 x the (hi, lo) pair of -mref, so its result starts the scores at -mref; mref is kept at values the
    // pair holds exactly
    const uint32_t onew = h2 == 0 ? 0x3C003C00u : 0u;
    const pa_u2 dcw = h2 == 0 ? (pa_u2){dcb[0], dcb[1]} : (pa_u2){dcb[2], dcb[3]};
    uint32_t mcw = 0u;
    // EX: the integer dots' start value, whose sum with a dot is the bits of the float 1.5 * 2^23 + dot (|dot| < 2^21): a
    // subtraction then converts it exactly, at twice the rate of v_cvt_f32_i32 (1.0 against 1.8 ns per wave instruction
    // and SIMD with two waves)
    mm_i16 cvt0;
    #pragma unroll
    for (int v = 0; v < 16; v++) cvt0[v] = 0x4B400000;
    if constexpr (EX && HD == 128) asm volatile("" : "+v"(cvt0));         // kept in registers, not rebuilt for every tile

    // ---- prologue: tile t0 -> stage 0, tile t0 + 2's loads in flight in R0 (t0 + 1's in R1)
    store_tile(R0, 0);
    load_tile(R0, PF);
    mm_lds_barrier();

    mm_f16 O[NBLK];
    #pragma unroll
    for (int db = 0; db < NBLK; db++) O[db] = (mm_f16){};
    float mref = -INFINITY, mx = -INFINITY, lsum = 0.0f;
    const float sm = a.qmode == 0 && FMT == 0 ? a.scale * MM_LOG2E : MM_LOG2E;   // score -> base-2 logit (!EX)
    float mc = 0.0f;                                                 // EX: mref once it is finite (0 before), the shift
                                                                     // the block dots start from
    const mm_h2 one2 = {(_Float16) 1.0f, (_Float16) 1.0f};
    const bool own = a.own_ref != 0;
    const float pmax = own ? -INFINITY : MM_PMAX;

    const int q4 = lane >> 4, s4 = lane & 15;
    // a tile's K operands (A operand of S^T, lane (h2, n): key n; !EX: dims 16kk + 8h2 .. +7; EX: the quants of dims 32b +
    // 16h2 .. +15 and the scales of blocks 2 h2, 2 h2 + 1)
    constexpr int KA = HD == 128 ? 8 : FMT == 0 ? 2 : 3;              // !EX: K operands read ahead (of HD / 16)
    constexpr bool KEARLY = HD == 128 && !SKIP;                      // read before the staging (the registers allow it)
    mm_h8 kf[KA];
    pa_u4 kq[4];
    uint32_t dk2 = 0u;
    auto kf_read = [&](const char * Kt, int kk) { kf[kk % KA] = *(const mm_h8 *) (Kt + n * G::KST + 32 * kk + 16 * h2); };
    auto k_read = [&](int stage) {
        const char * Kt = smem + (stage * NS + sx) * G::STAGE;
        if constexpr (EX) {
            if constexpr (HD == 128) dk2 = *(const uint32_t *) (Kt + G::KT + G::VT + 8 * n + 4 * h2);
            #pragma unroll
            for (int b = 0; b < (HD == 128 ? 4 : 2); b++) kq[b] = *(const pa_u4 *) (Kt + n * G::KST8 + 32 * b + 16 * h2);
        } else {
            #pragma unroll
            for (int kk = 0; kk < KA; kk++) kf_read(Kt, kk);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // one tile's matrix work on LDS stage `stage` (nvalid keys)
    auto compute = [&](int stage, int nvalid) {
        const char * Kt = smem + (stage * NS + sx) * G::STAGE;
        const char * Vt = Kt + G::KT;

        // V^T per (dim block db, 16-key half mi), idx = 2 db + mi, by two transposing reads (lane 16q + s reads key row 16mi +
        // (8 for the second read) + 4(q >> 1) + s / 4, dims 32db + 16(q & 1) + 4(s % 4) .. +3). Head dim 128 holds all of
        // them, read under the QK MFMAs and the softmax; head dim 256 reads VA ahead
        constexpr int VA = HD == 128 ? 8 : 2;
        if constexpr (!KEARLY) k_read(stage);
        mm_f16 S = (mm_f16){};
        mm_h8 va[VA];
        auto v_read = [&](int idx) {
            const int db = idx >> 1, mi = idx & 1;
            const char * vb = Vt + (16 * mi + 4 * (q4 >> 1) + (s4 >> 2)) * G::VST + 2 * (32 * db + 16 * (q4 & 1) + 4 * (s4 & 3));
            const pa_h4 x0 = __builtin_bit_cast(pa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((MM_LDS mm_tr4 *) vb));
            const pa_h4 x1 = __builtin_bit_cast(pa_h4, __builtin_amdgcn_ds_read_tr16_b64_v4f16((MM_LDS mm_tr4 *) (vb + 8 * G::VST)));
            va[idx % VA] = __builtin_shufflevector(x0, x1, 0, 1, 2, 3, 4, 5, 6, 7);
        };
        if constexpr (EX && HD == 256) {
            // per block: the integer dot, then dot * dq_b(row) * dk_b(key) in fp32, the scales of this lane's 16 keys read from
            // the tile (in fp32, four keys per read): no registers for a scale product or a start value here. q4_0 quants
            // are staged as 16 (n - 8), their byte's high nibble, and dq_b is divided by 16.
            #pragma unroll
            for (int b = 0; b < NBLK; b++) {
                pa_f4 dk[4];
                #pragma unroll
                for (int j = 0; j < 4; j++) dk[j] = *(const pa_f4 *) (Kt + G::KT + G::VT + 4 * (32 * b + 8 * j + 4 * h2));
                const mm_i16 T = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(mm_i4, kq[b & 1]), __builtin_bit_cast(mm_i4, Qi[b]),
                                                                     (mm_i16){}, 0, 0, 0);
                if (b + 2 < NBLK) kq[b & 1] = *(const pa_u4 *) (Kt + n * G::KST8 + 32 * (b + 2) + 16 * h2);
                const float dq = __builtin_bit_cast(float, dqb[b]);
                #pragma unroll
                for (int v = 0; v < 16; v++) S[v] = fmaf((float) T[v] * dq, dk[v / 4][v % 4], b == 0 ? -mc : S[v]);
                __builtin_amdgcn_sched_barrier(0);
            }
            #pragma unroll
            for (int i = 0; i < VA; i++) v_read(i);
        } else if constexpr (EX) {
            // per block: the integer dot on the int8 matrix cores (A: key n's quants, dims 32b + 16h2 .. +15, read raw
            // from the tile; B: the query quants), the scale product, and dot * product summed in fp32
            const pa_u2 dkw = {pa_perm(0u, dk2, 0x01000100u), pa_perm(0u, dk2, 0x03020302u)};
            if constexpr (FMT == 2) {
                // q4_0: the scores start at -mref plus sum_b dk_b(key) * (-8 * qsum_b * dq_b)(row), one MFMA over the
                // blocks' (hi, lo) pairs and -mref, so that the unsigned nibble dots need no per-score offset
                S = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mm_h8, (pa_u4){dkw.x, dkw.y, onew, 0u}),
                                                           __builtin_bit_cast(mm_h8, (pa_u4){dcw.x, dcw.y, mcw, 0u}),
                                                           (mm_f16){}, 0, 0, 0);
            }
            #pragma unroll
            for (int b = 0; b < 4; b++) {
                const mm_f16 T = __builtin_bit_cast(mm_f16, __builtin_amdgcn_mfma_i32_32x32x32_i8(
                    __builtin_bit_cast(mm_i4, kq[b]), __builtin_bit_cast(mm_i4, Qi[b]), cvt0, 0, 0, 0));
                const mm_f16 Pb = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(pa_h4, dkw), __builtin_bit_cast(pa_h4, dqw[b]),
                                                                       (mm_f16){}, 0, 0, 0);
                #pragma unroll
                for (int v = 0; v < 16; v++) S[v] = fmaf(Pb[v], T[v] - 12582912.0f, b == 0 && FMT == 1 ? -mc : S[v]);
                __builtin_amdgcn_sched_barrier(0);
            }
            #pragma unroll
            for (int i = 0; i < VA; i++) v_read(i);                  // V^T after the block dots, under the softmax
        } else {
            // S^T = K Q'^T; at head dim 128 each MFMA is followed by the two transposing V reads of one (dim block, key half),
            // so that at most 15 LDS reads are outstanding (the counter's range) and each MFMA waits for its own K read only
            #pragma unroll
            for (int kk = 0; kk < HD / 16; kk++) {
                S = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[kk % KA], Qf[kk], S, 0, 0, 0);
                if (kk + KA < HD / 16) kf_read(Kt, kk + KA);
                if (kk >= HD / 16 - VA) v_read(kk - (HD / 16 - VA));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (nvalid < 32) {                                           // keys 8j + 4h2 + i past the page's end
            #pragma unroll
            for (int v = 0; v < 16; v++)
                if (8 * (v / 4) + 4 * h2 + (v % 4) >= nvalid) S[v] = -INFINITY;
        }
        float tm = fmaxf(fmaxf(S[0], S[1]), S[2]);                   // this lane's half of row n's tile max
        {
            const float t1 = fmaxf(fmaxf(S[3], S[4]), S[5]), t2 = fmaxf(fmaxf(S[6], S[7]), S[8]), t3 = fmaxf(fmaxf(S[9], S[10]), S[11]),
                        t4 = fmaxf(fmaxf(S[12], S[13]), S[14]);
            tm = fmaxf(fmaxf(fmaxf(tm, t1), t2), fmaxf(fmaxf(t3, t4), S[15]));
        }
        tm = EX ? tm + mc : tm * sm;                                 // base 2
        if (__builtin_amdgcn_ballot_w64(tm > mref + pmax)) {
            // rare: move the reference max of every row that needs it (uniform branch); own_ref: to every tile's maximum
            const float tr = mm_max32(tm);                           // the row's other half: lane ^ 32
            float mn = own ? fmaxf(tr, mm_max32(fmaxf(mx, tm)) - MM_OWN) : fmaxf(mref, tr);
            if constexpr (EX && FMT == 2 && HD == 128) {             // a value the (hi, lo) pair of -mn holds exactly
                const _Float16 mh = (_Float16) mn, ml = (_Float16) (mn - (float) mh);
                mn = (float) mh + (float) ml;
                const _Float16 nh = -mh, nl = -ml;
                mcw = h2 == 0 ? (uint32_t) __builtin_bit_cast(uint16_t, nh) | ((uint32_t) __builtin_bit_cast(uint16_t, nl) << 16) : 0u;
            }
            const float alpha = mref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mref - mn);
            #pragma unroll
            for (int db = 0; db < NBLK; db++) O[db] *= alpha;
            lsum *= alpha;
            mref = mn;
            if constexpr (EX) {                                      // rebase this tile's scores and the start value
                const float dl = mn - mc;
                #pragma unroll
                for (int v = 0; v < 16; v++) S[v] -= dl;
                mc = mn;
            }
        }
        mx = fmaxf(mx, tm);
        mm_h8 P[2];
        #pragma unroll
        for (int v = 0; v < 16; v++)
            P[v / 8][v % 8] = (_Float16) __builtin_amdgcn_exp2f(EX ? S[v] : fmaf(S[v], sm, -mref));
        #pragma unroll
        for (int v = 0; v < 16; v += 2) {                            // the row sum of the fp16 P the PV MFMAs use
            const mm_h2 pp = {P[v / 8][v % 8], P[v / 8][v % 8 + 1]};
            lsum = __builtin_amdgcn_fdot2(pp, one2, lsum, false);
        }

        // ---- O^T += V^T P^T
        #pragma unroll
        for (int i = 0; i < 2 * NBLK; i++) {
            O[i >> 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[i % VA], P[i & 1], O[i >> 1], 0, 0, 0);
            if (i + VA < 2 * NBLK) v_read(i + VA);
        }
    };
    // one tile step; Rn holds tile t + 1's raw bytes
    auto step = [&](uint32_t t, MmRaw<FMT> (&Rn)[NS][UPT]) {
        const int stage = t & 1;
        int nvalid = 0;                                              // keys of this wave's tile (0 past the chunk's end)
        #pragma unroll
        for (int x = 0; x < NS; x++) {
            if (NS > 1 && NS * t + x >= ntiles) break;
            if (ctl == 0) {                                          // before any LDS operation of this step
                uint32_t keys;
                do { cpg++; keys = a.pstart[cpg + 1] - a.pstart[cpg]; } while (keys == 0);
                ctl = (keys - 1) / 32 + 1;
                clast = (keys - 1) % 32 + 1;
                __builtin_amdgcn_s_waitcnt(0xc07f);
            }
            const uint32_t nv = ctl == 1 ? clast : 32u;
            ctl -= 1;
            if (NS == 1 || x == sx) nvalid = (int) nv;
        }
        const bool clive = wlive && (NS == 1 || nvalid > 0);
        // the next step's bytes -> the other stage (last read before the previous barrier; past the chunk's end the
        // stage is written and never read), then step t + 1 + PF's loads into the registers just freed
        if (KEARLY) k_read(stage);
        store_tile(Rn, stage ^ 1);
        load_tile(Rn, t + 1 + PF);
        if (clive) compute(stage, nvalid);
        mm_lds_barrier();                                            // this stage is free; the next one is written
    };
    const uint32_t nsteps = (ntiles + NS - 1) / NS;
    uint32_t t = 0;                                                  // step t + 1's tiles are in R((t + 1) % PF)
    if constexpr (PF == 2) {
        for (; t + 2 <= nsteps; t += 2) {
            step(t, R1);
            step(t + 1, R0);
        }
        if (t < nsteps) step(t, R1);
    } else {
        for (; t < nsteps; t++) step(t, R0);
    }

    if constexpr (NS > 1) {
        // fold the streams: each but the first leaves its rows' O, reference and exact max and sum in the stages (free after
        // the last barrier), lane by lane; the first one's waves rebase both to the larger reference max and add
        float * fold = (float *) smem + rw * 67 * 64 + lane;
        static_assert(RW * 67 * 256 <= 2 * NS * G::STAGE, "the streams fold through the stages");
        #pragma unroll
        for (int x = 1; x < NS; x++) {
            if (sx == x && wlive) {
                #pragma unroll
                for (int db = 0; db < NBLK; db++)
                    #pragma unroll
                    for (int v = 0; v < 16; v++) fold[64 * (16 * db + v)] = O[db][v];
                fold[64 * 64] = mref; fold[64 * 65] = mx; fold[64 * 66] = lsum;
            }
            mm_lds_barrier();
            if (sx == 0 && wlive) {
                const float m1 = fold[64 * 64], mn = fmaxf(mref, m1);
                const float f0 = mref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mref - mn);
                const float f1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mn);
                #pragma unroll
                for (int db = 0; db < NBLK; db++)
                    #pragma unroll
                    for (int v = 0; v < 16; v++) O[db][v] = O[db][v] * f0 + fold[64 * (16 * db + v)] * f1;
                mx = fmaxf(mx, fold[64 * 65]);
                lsum = lsum * f0 + fold[64 * 66] * f1;
                mref = mn;
            }
            if (x + 1 < NS) mm_lds_barrier();
        }
        if (sx != 0) return;
    }
    mx = mm_max32(mx);                                               // the exact row max, tracked per half row
    mm_write_out<HD>(a, O, mref, mx, lsum, h, row, rlive, h2, c);
}

// The ggml query rounding over quantized K takes the exact block dots at every size (4-wave verify blocks and 8-wave
// prefill chunks); the reference engines' rounding (PA_QMODE_F16) and f16 K take the fp16-operand QK, the Metal
// engine's own arithmetic (K dequantized to half in threadgroup memory, pa-metal.mm:379-487)
template <int HD, int FMT, bool EX>
static hipError_t launch_mma_fmt(int nw, bool skip, int streams, const AttnArgs & a, uint32_t grid, hipStream_t st, hipEvent_t ev0,
                                 hipEvent_t ev1) {
    switch (nw) {
        case 4:
            if (streams == 2) hipExtLaunchKernelGGL((mma_kernel<128, FMT, 4, true, EX, 2>), dim3(grid), dim3(256), 0, st, ev0, ev1, 0, a);
            else if (skip) hipExtLaunchKernelGGL((mma_kernel<HD, FMT, 4, true, EX>), dim3(grid), dim3(256), 0, st, ev0, ev1, 0, a);
            else hipExtLaunchKernelGGL((mma_kernel<HD, FMT, 4, false, EX>), dim3(grid), dim3(256), 0, st, ev0, ev1, 0, a);
            break;
        case 8:
            if (skip) hipExtLaunchKernelGGL((mma_kernel<HD, FMT, 8, true, EX>), dim3(grid), dim3(512), 0, st, ev0, ev1, 0, a);
            else hipExtLaunchKernelGGL((mma_kernel<HD, FMT, 8, false, EX>), dim3(grid), dim3(512), 0, st, ev0, ev1, 0, a);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static hipError_t launch_mma_128(int fmt, int nw, bool skip, int streams, const AttnArgs & a, uint32_t grid, hipStream_t st, hipEvent_t ev0,
                                 hipEvent_t ev1) {
    const bool ex = a.qmode == 0;                                    // PA_QMODE_GGML over quantized K: exact block dots
    if (fmt == 0) return launch_mma_fmt<128, 0, false>(nw, skip, streams, a, grid, st, ev0, ev1);
    if (fmt == 1) return ex ? launch_mma_fmt<128, 1, true>(nw, skip, streams, a, grid, st, ev0, ev1) : launch_mma_fmt<128, 1, false>(nw, skip, streams, a, grid, st, ev0, ev1);
    if (fmt == 2) return ex ? launch_mma_fmt<128, 2, true>(nw, skip, streams, a, grid, st, ev0, ev1) : launch_mma_fmt<128, 2, false>(nw, skip, streams, a, grid, st, ev0, ev1);
    return hipErrorInvalidValue;
}

// (the exact block dots at head dim 256 are taken above 512 rows only: every wave of one of their row blocks at least has rows)
template <int FMT, bool EX>
static hipError_t launch_mma_256_fmt(bool skip, const AttnArgs & a, uint32_t grid, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    if (!skip) hipExtLaunchKernelGGL((mma_kernel<256, FMT, 8, false, EX>), dim3(grid), dim3(512), 0, st, ev0, ev1, 0, a);
    else if constexpr (!EX) hipExtLaunchKernelGGL((mma_kernel<256, FMT, 8, true, EX>), dim3(grid), dim3(512), 0, st, ev0, ev1, 0, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

static hipError_t launch_mma_256(int fmt, bool skip, const AttnArgs & a, uint32_t grid, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1) {
    const bool ex = a.qmode == 0;
    if (fmt == 0) return launch_mma_256_fmt<0, false>(skip, a, grid, st, ev0, ev1);
    if (fmt == 1) return ex ? launch_mma_256_fmt<1, true>(skip, a, grid, st, ev0, ev1) : launch_mma_256_fmt<1, false>(skip, a, grid, st, ev0, ev1);
    if (fmt == 2) return ex ? launch_mma_256_fmt<2, true>(skip, a, grid, st, ev0, ev1) : launch_mma_256_fmt<2, false>(skip, a, grid, st, ev0, ev1);
    return hipErrorInvalidValue;
}

hipError_t launch_mma(int hd, int fmt, int nw, bool skip, int streams, const AttnArgs & a, uint32_t grid, hipStream_t st, hipEvent_t ev0,
                      hipEvent_t ev1) {
    if (hd == 128) return launch_mma_128(fmt, nw, skip, streams, a, grid, st, ev0, ev1);
    if (hd == 256 && nw == 8) return launch_mma_256(fmt, skip, a, grid, st, ev0, ev1);
    return hipErrorInvalidValue;
}

}  // namespace pa_hip
