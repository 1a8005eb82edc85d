// sdpa_prefill.hip -- causal attention over a whole prompt (prefill) for gfx950, on bf16 MFMA.
//
//   O[s, h] = softmax_{t <= s}(q[s, h] . k[t, kv(h)] / sqrt(128)) . v[t, kv(h)],  kv(h) = h / (H / H_KV)
//
// The contract of the reference's sdpa_prefill_bf16 (nemotron_infer/csrc/include/ops/attention/
// sdpa_prefill.cuh:224-320, host entry :364-395): causal, GQA, head dim 128, float32 softmax and
// accumulation on bf16 inputs, bf16 output.  The layouts are this build's: q, k, v and O stay
// token-major ([S, heads * 128], as the projections write them) -- the reference transposes
// them to head-major around its kernel (model/attention_block.cuh:339-345); V is read token-major
// too, its MFMA operand built by transposing LDS reads.
//
// Kernel: one workgroup per (query head, tile of 128 query rows), 4 waves of 32 rows.  K and V
// reach LDS by DMA (global_load_lds_dwordx4, no register staging), token-major and swizzled so
// that the operand reads hit distinct banks: K in blocks of 32 keys (four 8 KiB slots), V in tiles
// of 64 keys (two 16 KiB stages); one barrier per 64 keys.  Per wave and 32-key block
// (v_mfma_f32_32x32x16_bf16):
// * S^T = K . Q^T (32 keys x 32 queries): the wave's query rows are the B operand, held in
//   registers for the whole kernel; the scores of one query then sit in one lane (16 registers,
//   the two lane halves holding alternate 4-key groups), so the row max and sum are in-lane, with
//   one exchange between the halves per block for the max and one at the end for the sum.
// * online softmax in base 2 (weights exp2((s - m) log2(e) / sqrt(128)) with one fma per score),
//   the running max m raised lazily (only when a score exceeds it by 2^8 in weight, so the
//   accumulators are rescaled rarely); keys after the query masked on the diagonal blocks only.
// * O^T += V^T . P^T: P is the B operand straight from the score registers -- a 16-key step's
//   lane-half h holds keys {4h..4h+3, 8+4h..8+4h+3} -- in two bf16 parts (hi = bf16(p), lo =
//   bf16(p - hi)), so the weights carry about 16 significant bits.  The row sum is float32: a block's
//   16 weights in a lane first, then one add per block, so that its error grows with the blocks and
//   not with the keys (one running sum over all keys was off by 6e-5 in a flat row of 8192, this
//   by 2e-6).  The V^T operand, in the same key order, comes from two transposing
//   LDS reads (ds_read_b64_tr_b16) of the token-major V tile.
// The three run as a pipeline over blocks: while the matrix cores do the products with V of block g
// and the scores of block g + 2, the same wave's vector unit turns the scores of block g + 1 into
// weights.  A 32-cycle MFMA hides up to six vector instructions or two exponentials of its own
// wave (measured), so the 24 MFMAs of a block are laid out in 24 slots with the block's 106 vector
// instructions and 24 LDS reads spread over them; the compiler's own order ran the vector work
// between the MFMAs' blocks.  Times beside that form (scores one block ahead, weights in
// the block that uses them), 40 / 8 heads, S = 512 / 1000 / 2048 / 4096 / 8192: 17.5 / 31.4 / 69.8
// / 235.9 / 877.5 -> 16.2 / 27.9 / 65.5 / 223.6 / 826.9 us; 16 / 4 heads, S = 2048: 52.4 -> 43.7.
// At S = 4096 the cycles fell by 16% and the clock with them (2.1 -> 1.76 GHz): with the matrix
// cores busy 62% of the time at 1.5 times the plain flops (P in two parts) the power budget is the
// next bound.
// The last tile has a body of its own without the scores that nothing follows (40 / 8 heads, S = 1 /
// 33 / 64 / 192: 4.7 / 5.6 / 6.0 / 8.8 -> 4.2 / 4.7 / 5.4 / 8.3 us): with them the short prompts were
// slower than in the form above (4.9 / 5.3 / 5.9 / 9.1).  65 to 128 tokens still are, by 0.1 to 0.4 us
// (S = 128 7.7 / 8.1): two tiles are too few to pay for filling the pipeline.
// The KV caches of the attention block are filled by the same launch (it was one of its own, 5-7 us).
// Query tiles are scheduled longest first over all heads (the last tiles see the most keys).
#include "nmi_device.hpp"
#include "nmi_launch.hpp"

#include <cfloat>
#include <type_traits>

namespace nmi {

namespace {

constexpr int kD = 128;           // head dim
constexpr int kBQ = 128;          // query rows per workgroup
constexpr int kBK = 64;           // key positions per tile
constexpr int kKBlk = 32 * kD * 2;           // K block of 32 keys, 8 KiB (four slots)
constexpr int kVBytes = kBK * kD * 2;        // V tile of 64 keys, 16 KiB (two stages)
constexpr int kLds = 4 * kKBlk + 2 * kVBytes;
constexpr float kLazy = 8.f;       // log2 of the largest unnormalised softmax weight (lazy max)

struct PrefillArgs {
    const uint16_t* q;      // [S, ldq], head h at column 128 h
    const uint16_t* k;      // [S, ldk], KV head j at column 128 j
    const uint16_t* v;      // [S, ldv], KV head j at column 128 j
    uint16_t* o;            // [S, ldo], head h at column 128 h
    int64_t ldq, ldk, ldv, ldo;
    int S, H, H_KV, qtiles;
    int nslot;              // workgroups per pass of the dispatcher (one per CU)
    float scale2;           // log2(e) / sqrt(128)
    float lazy;             // kLazy / scale2
    uint16_t* k_cache;      // [H_KV, cap, 128] caches to fill from k and v (positions [0, S)), or nullptr
    uint16_t* v_cache;
    int cap;
};

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// LDS K tile: row r (key) of 16 chunks of 16 B, chunk c at c ^ (r & 15)
__device__ __forceinline__ int k_off(int r, int c) { return r * 256 + ((c ^ (r & 15)) << 4); }
typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4i16 lds_v4i16;

__global__ __launch_bounds__(256, 2) void sdpa_prefill_kernel(const PrefillArgs a) {
    typedef __attribute__((address_space(3))) void lds_void;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void*)lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, l32 = lane & 31;
    // Tiles by rank, longest first over all heads: rank r is query tile qtiles - 1 - r / H of head
    // r % H.  The dispatcher gives each CU one workgroup per pass (workgroups g and g + nslot
    // share a CU), so the second pass takes its ranks in reverse: a CU then holds a long and a
    // short tile of about the same sum; the rest follow longest first.
    const int total = a.qtiles * a.H, g = (int)blockIdx.x;
    const int n2 = min(2 * a.nslot, total);
    const int rank = (g >= a.nslot && g < n2) ? a.nslot + (n2 - 1 - g) : g;
    const int qt = a.qtiles - 1 - rank / a.H;
    const int head = rank - rank / a.H * a.H;
    const int kvh = head / (a.H / a.H_KV);
    const int q0 = qt * kBQ;
    const int qw = q0 + 32 * wave;                              // the wave's first query row
    const int qrow = qw + l32;                                  // this lane's query (B operand column)
    const int S = a.S;
    const int kv_end = min(S, q0 + kBQ);                        // keys this workgroup needs
    const int ntiles = (kv_end + kBK - 1) / kBK;

    // the wave's query rows as B fragments: k step s holds dims 16 s + 8 h .. + 7 of row qrow
    bf16x8 qf[8];
    {
        const uint16_t* qp = a.q + (int64_t)min(qrow, S - 1) * a.ldq + head * kD + 8 * h;
#pragma unroll
        for (int s = 0; s < 8; ++s) qf[s] = __builtin_bit_cast(bf16x8, load16(qp + 16 * s));
    }

    // LDS: K blocks of 32 keys, block g in slot g % 4 at g % 4 * 8 KiB; V tiles of 64 keys, tile t in
    // stage t & 1 at 32 KiB + (t & 1) * 16 KiB; both token-major, 256 B per key.
    // LDS DMA sources.  Instruction i of the wave fills rows r = 16 i + 4 wave + lane / 16 of a K slot
    // (i = 0, 1) or V stage (i = 0 .. 3) (1 KiB: 4 rows of 256 B); lane position p = lane % 16 of row r
    // takes chunk p ^ (r & 15) (K) or p ^ (4 (r & 3)) (V).  The swizzles do not depend on i, so one
    // lane offset serves every instruction (i moves the scalar base).
    const int64_t ldk2 = a.ldk * 2, ldv2 = a.ldv * 2;
    const int kr0 = 4 * wave + (lane >> 4);
    const uint32_t kchunk = 16u * (uint32_t)((lane & 15) ^ (kr0 & 15));
    const uint32_t koff = (uint32_t)(kr0 * ldk2) + kchunk;
    const uint32_t vchunk = 16u * (uint32_t)((lane & 15) ^ (4 * (kr0 & 3)));
    const uint32_t voff = (uint32_t)(kr0 * ldv2) + vchunk;
    const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.k + kvh * kD);
    const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.v + kvh * kD);
    const int nblk = 2 * ntiles;
    // K block g into slot g % 4; rows past S - 1 (of a last, partial block, or of a block wholly
    // past S) read row S - 1
    auto issue_k = [&](int g) {
        const int kv0 = 32 * g;
        const uint32_t sb = lds0 + (uint32_t)((g & 3) * kKBlk) + wave * 1024;
        if (kv0 + 32 <= S) {
            const uint8_t* base = kbase + (int64_t)kv0 * ldk2;
#pragma unroll
            for (int i = 0; i < 2; ++i) dma16_lds(base + 16 * i * ldk2, koff, sb + i * 4096);
        } else {
            const int r0 = min(kv0, S - 1);
            const uint8_t* base = kbase + (int64_t)r0 * ldk2;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                dma16_lds(base, (uint32_t)((min(kv0 + 16 * i + kr0, S - 1) - r0) * ldk2) + kchunk, sb + i * 4096);
        }
    };
    // V tile t (64 keys, token-major) into stage t & 1, row r's chunk c at c ^ (4 (r & 3)); rows past
    // S - 1 read row S - 1 (finite values; their weights are 0)
    auto issue_v = [&](int t) {
        const int kv0 = t * kBK;
        const uint32_t sb = lds0 + (uint32_t)(4 * kKBlk + (t & 1) * kVBytes) + wave * 1024;
        if (kv0 + kBK <= S) {
            const uint8_t* base = vbase + (int64_t)kv0 * ldv2;
#pragma unroll
            for (int i = 0; i < 4; ++i) dma16_lds(base + 16 * i * ldv2, voff, sb + i * 4096);
        } else {
            const int r0 = min(kv0, S - 1);
            const uint8_t* base = vbase + (int64_t)r0 * ldv2;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                dma16_lds(base, (uint32_t)((min(kv0 + 16 * i + kr0, S - 1) - r0) * ldv2) + vchunk, sb + i * 4096);
        }
    };
    // V^T operand reads (ds_read_b64_tr_b16: in each 16-lane group, output lane 4 a + b, element e
    // is element b of source lane 4 e + a's 8 bytes).  For key step j, dim block b and part q,
    // source lane s of group G reads key row 16 j + 8 q + 4 (G / 2) + s / 4, dims 32 b + 16 (G % 2)
    // + 4 (s % 4) .. + 3; lane (l32, h) then holds keys 16 j + 8 q + 4 h + {0..3} of dim 32 b + l32
    // -- the P operand's key order.  Per lane: the byte offset within a stage of part 0 of key step
    // 0 for each b (key step and part add 4096 j + 2048 q).
    uint32_t vtr[4];
    {
        const int G = lane >> 4, s16 = lane & 15;
        const int rb = 4 * (G >> 1) + (s16 >> 2);
        const int cb = 2 * (G & 1) + ((s16 & 3) >> 1);
#pragma unroll
        for (int b = 0; b < 4; ++b)
            vtr[b] = (uint32_t)(rb * 256 + 64 * (b ^ (rb & 3)) + 16 * cb + 8 * (s16 & 1));
    }

    f32x16 oacc[4];                                             // O^T: 4 blocks of 32 dims x 32 queries
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[b][r] = 0.f;
    float m = -INFINITY, l = 0.f;       // raw score units; l is this lane half's share of the row sum
    float corr = 1.f;                   // oacc's pending rescale
    bool pending = false;               // (wave-uniform)

    // causal mask of a block of 32 keys at kvb (only where it reaches past the wave's first query):
    // register r is key kvb + 8 (r / 4) + 4 h + r % 4, kept where it is <= qrow, then also < S for
    // every stored query
    auto mask = [&](f32x16& sc, int kvb) {
        if (kvb + 31 > qw) {
            // a branch the compiler keeps: the blocks below the diagonal skip the mask entirely
            asm volatile("" ::: "memory");
            const int dq = qrow - kvb - 4 * h;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (8 * (r >> 2) + (r & 3) > dq) sc[r] = -INFINITY;
        }
    };
    // The running max m raised lazily by a block's in-lane max: only when a score exceeds it by more
    // than 8 / scale2 (the weights exp2((s - m) scale2) stay below 2^8).  O / l does not depend on
    // m.  The first block holds key 0, so every query's max is finite from there on.  l holds the
    // earlier blocks and is rescaled at once; oacc still misses the block before, whose weights are
    // under the old max, and is rescaled after that block's products (settle).
    auto raise_max = [&](float tmax) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(tmax), __float_as_uint(tmax), false, false);
        tmax = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));       // both lane halves
        const bool raise = tmax > m + a.lazy;
        if (__builtin_amdgcn_ballot_w64(raise)) {
            const float mn = raise ? tmax : m;
            corr = raise ? fexp2((m - mn) * a.scale2) : 1.f;
            l *= corr;
            m = mn;
            pending = true;
        }
    };
    auto settle = [&]() {
        if (pending) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[b][r] *= corr;
            pending = false;
        }
    };
    auto row_max = [&](const f32x16& sc) {
        float t = sc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) t = fmaxf(t, sc[r]);
        return t;
    };
    // The weights of 16 scores as the P^T B fragments of key steps 0 and 1 (registers 8 j .. + 7), each
    // in two bf16 parts: hi = bf16(p), lo = bf16(p - hi).  Three stages per pair of scores e = 2 i,
    // 2 i + 1, so that a pair can be spread over three MFMAs.
    struct Weights {
        uint32_t hi[8], lo[8];
    };
    float p0 = 0.f, p1 = 0.f;
    float psum = 0.f;                   // the 16 weights' sum, added to l by their block (see below)
    // pin: keeps the computation of x in the slot it is written in (the compiler otherwise sinks it
    // to the block that uses it, past all the MFMAs meant to hide it)
    auto pin = [](auto& x) __attribute__((always_inline)) { asm volatile("" : "+v"(x)); };
    auto weigh = [&](const f32x16& sc, float mc, int i, int stage, Weights& w) __attribute__((always_inline)) {
        if (stage == 0) {
            p0 = fexp2(__builtin_fmaf(sc[2 * i], a.scale2, -mc));
            p1 = fexp2(__builtin_fmaf(sc[2 * i + 1], a.scale2, -mc));
            pin(p0);
            pin(p1);
        } else if (stage == 1) {
            w.hi[i] = pack_bf16(p0, p1);
            psum = i == 0 ? p0 + p1 : psum + p0 + p1;
            pin(w.hi[i]);
            pin(psum);
        } else {
            // (v_dot2 would save the unpacking of hi, but beside MFMAs each costs 16 cycles and more)
            w.lo[i] = pack_bf16(p0 - bf16lo_to_f32(w.hi[i]), p1 - bf16hi_to_f32(w.hi[i]));
            pin(w.lo[i]);
        }
    };
    auto frag = [&](const uint32_t (&w)[8], int j) {
        return __builtin_bit_cast(bf16x8, uint4{w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]});
    };
    auto read_k = [&](const uint8_t* kst, int s) {
        return *reinterpret_cast<const bf16x8*>(kst + k_off(l32, 2 * s + h));
    };
    auto read_v = [&](const uint8_t* vst, int j, int b) {
        const v4i16 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vst + vtr[b] + 4096 * j));
        const v4i16 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)(vst + vtr[b] + 4096 * j + 2048));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // Block g (32 keys: key steps j0, j0 + 1 of the V tile at vst) of a three-deep pipeline: the 16
    // products O^T += V^T . P^T of block g (weights wc), the 8 products S^T = K . Q^T of block g + 2
    // (K slot at kst, into nxt), and the weights of block g + 1 (scores sc, into wn).  None of the
    // three depends on another within the block, so the matrix cores run under the vector work of the
    // same wave: 24 slots of one MFMA, at most two LDS reads (three slots ahead of their use) and
    // three or four vector instructions, fenced so that the compiler keeps them apart.  Then block
    // g + 2's mask and max.  kvb2: its first key.
    auto block = [&](auto masked, const f32x16& sc, f32x16& nxt, const Weights& wc, Weights& wn, const uint8_t* kst,
                     const uint8_t* vst, int j0, int kvb2) __attribute__((always_inline)) {
        const float mc = m * a.scale2;
        bf16x8 kf[4], vf[3];
        kf[0] = read_k(kst, 0);
        kf[1] = read_k(kst, 1);
        vf[0] = read_v(vst, j0, 0);
        weigh(sc, mc, 0, 0, wn);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) nxt[r] = 0.f;
        float tmax = 0.f;
#pragma unroll
        for (int q = 0; q < 24; ++q) {
            // MFMA: S in slots 0, 1, 3, 4, 6, 7, 9, 10; P.V (hi, lo of each V fragment u) in the others
            const bool is_k = q < 11 && q % 3 != 2;
            if (is_k) {
                const int st = 2 * (q / 3) + q % 3;
                nxt = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[st & 3], qf[st], nxt, 0, 0, 0);
                if (st + 2 < 8) kf[(st + 2) & 3] = read_k(kst, st + 2);
            } else {
                const int p = q < 12 ? q / 3 : q - 8, u = p >> 1, b = u & 3;
                const bf16x8 w = frag((p & 1) ? wc.lo : wc.hi, u >> 2);
                oacc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u % 3], w, oacc[b], 0, 0, 0);
            }
            // V fragment u + 1: at slot 4 (u = 0), then three or four slots ahead of its use
            if (q == 4) vf[1] = read_v(vst, j0, 1);
            if (q >= 9 && q <= 19 && (q & 1)) {
                const int u = (q - 9) / 2 + 2;
                vf[u % 3] = read_v(vst, j0 + (u >> 2), u & 3);
            }
            // vector work: pair q / 3's stages (pair 0's first is above), one stage ahead of the slot
            if (q < 23) weigh(sc, mc, (q + 1) / 3, (q + 1) % 3, wn);
            if constexpr (!decltype(masked)::value) {
                if (q == 14) tmax = fmaxf(fmaxf(nxt[0], nxt[1]), nxt[2]);
                if (q >= 15 && q <= 20) tmax = fmaxf(fmaxf(tmax, nxt[2 * q - 27]), nxt[2 * q - 26]);
                if (q == 21) tmax = fmaxf(tmax, nxt[15]);
                if (q >= 14 && q <= 21) pin(tmax);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (decltype(masked)::value) {
            mask(nxt, kvb2);
            tmax = row_max(nxt);
        }
        l += psum;                      // block g + 1's, still under the max its weights were formed with
        settle();
        raise_max(tmax);
    };
    // The same for the last tile, after which no scores are needed: the products with V of block g
    // (weights wc) and, with weighs, the weights of block g + 1.
    auto finish = [&](auto weighs, const f32x16& sc, const Weights& wc, Weights& wn, const uint8_t* vst,
                      int j0) __attribute__((always_inline)) {
        const float mc = m * a.scale2;
        bf16x8 vf[3];
        vf[0] = read_v(vst, j0, 0);
        vf[1] = read_v(vst, j0, 1);
#pragma unroll
        for (int p = 0; p < 16; ++p) {
            const int u = p >> 1, b = u & 3;
            const bf16x8 w = frag((p & 1) ? wc.lo : wc.hi, u >> 2);
            oacc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[u % 3], w, oacc[b], 0, 0, 0);
            if (!(p & 1) && u + 2 < 8) vf[(u + 2) % 3] = read_v(vst, j0 + ((u + 2) >> 2), (u + 2) & 3);
            if constexpr (decltype(weighs)::value) {
#pragma unroll
                for (int s = 24 * p / 16; s < 24 * (p + 1) / 16; ++s) weigh(sc, mc, s / 3, s % 3, wn);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (decltype(weighs)::value) l += psum;
        settle();
    };
    auto kslot = [&](int g) { return lds + (g & 3) * kKBlk; };
    auto vstage = [&](int t) { return lds + 4 * kKBlk + (t & 1) * kVBytes; };
    // Tile t = blocks 2 t, 2 t + 1.  On entry wa holds block 2 t's weights, sb block 2 t + 1's scores;
    // K slots hold blocks 2 t + 2 and 2 t + 3, V stage t & 1 tile t.  The DMAs refill the slots and
    // the stage read in tile t - 1 (published by its closing barrier).  P, the parity of t, makes the
    // LDS offsets constants.
    f32x16 sa, sb;
    Weights wa, wb;
    auto issue = [&](int t) {
        issue_v(t + 1);
        if (2 * t + 4 < nblk) {
            issue_k(2 * t + 4);
            issue_k(2 * t + 5);
        }
    };
    // this wave's DMAs done and its LDS reads returned (the compiler may place the MFMAs that consume
    // the last reads after this statement; the stages they read are refilled right after the
    // barrier), then the barrier
    auto publish = []() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    // below the diagonal: P, the parity of t, makes the LDS offsets constants
    auto step = [&](auto P, int t) __attribute__((always_inline)) {
        constexpr int par = decltype(P)::value;
        constexpr std::false_type masked{};
        issue(t);
        block(masked, sb, sa, wa, wb, kslot(2 * par + 2), vstage(par), 0, t * kBK + 64);
        block(masked, sa, sb, wb, wa, kslot(2 * par + 3), vstage(par), 2, t * kBK + 96);
        publish();
    };

    issue_k(0);
    issue_k(1);
    issue_v(0);
    if (nblk > 2) {
        issue_k(2);
        issue_k(3);
    }
    // K blocks 0 and 1 landed (the query's loads too, so the compiler has no load of its own
    // outstanding), then the barrier that publishes them; V tile 0 and K blocks 2, 3 may still be
    // on their way
#pragma unroll
    for (int s = 0; s < 8; ++s) asm volatile("" ::"v"(qf[s]));
    if (nblk > 2) asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(4)\n\ts_barrier" ::: "memory");
    // this workgroup's share of the KV cache fill: its own rows, by one query head of the group
    const bool fill = a.k_cache && head % (a.H / a.H_KV) == qt % (a.H / a.H_KV);
    uint4 kr[8], vr[8];
    if (fill) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int p = min(q0 + (tid >> 4) + 16 * u, S - 1);
            kr[u] = load16(a.k + (int64_t)p * a.ldk + kvh * kD + 8 * (tid & 15));
            vr[u] = load16(a.v + (int64_t)p * a.ldv + kvh * kD + 8 * (tid & 15));
        }
    }
    // fill the pipeline: scores of blocks 0 and 1, weights of block 0
#pragma unroll
    for (int r = 0; r < 16; ++r) sa[r] = sb[r] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_k(kslot(0), s), qf[s], sa, 0, 0, 0);
        sb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(read_k(kslot(1), s), qf[s], sb, 0, 0, 0);
    }
    if (fill) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int p = q0 + (tid >> 4) + 16 * u;
            if (p < S) {
                const int64_t off = ((int64_t)kvh * a.cap + p) * kD + 8 * (tid & 15);
                *reinterpret_cast<uint4*>(a.k_cache + off) = kr[u];
                *reinterpret_cast<uint4*>(a.v_cache + off) = vr[u];
            }
        }
    }
    mask(sa, 0);
    mask(sb, 32);
    raise_max(row_max(sa));
    settle();
    {
        const float mc = m * a.scale2;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int st = 0; st < 3; ++st) weigh(sa, mc, i, st, wa);
    }
    l += psum;
    raise_max(row_max(sb));
    // the rest landed; and slots 0 and 1 are refilled in tile 0: every wave's reads of them first
    publish();
    int t = 0;
    // tiles t, t + 1 compute the scores of keys up to 64 t + 255: below the diagonal while that is
    // before the workgroup's first query
    for (; t * kBK + 4 * kBK <= q0; t += 2) {
        step(std::integral_constant<int, 0>{}, t);
        step(std::integral_constant<int, 1>{}, t + 1);
    }
    // the last tiles (up to four) but the very last, one body for all.  Each wave takes the blocks
    // with a key <= some query of its own; the scores past those are masked.
    for (; t + 1 < ntiles; ++t) {
        issue(t);
        if (qw < S && t * kBK <= qw + 31) {
            constexpr std::true_type masked{};
            block(masked, sb, sa, wa, wb, kslot(2 * t + 2), vstage(t), 0, t * kBK + 64);
            if (t * kBK + 32 <= qw + 31) block(masked, sa, sb, wb, wa, kslot(2 * t + 3), vstage(t), 2, t * kBK + 96);
        }
        publish();
    }
    if (qw < S && t * kBK <= qw + 31) {
        int j0 = 0;
        if (t * kBK + 32 <= qw + 31) {
            finish(std::true_type{}, sb, wa, wb, vstage(t), 0);
            wa = wb;                    // (one body for the second half)
            j0 = 2;
        }
        finish(std::false_type{}, sb, wa, wb, vstage(t) + 4096 * j0, 0);
    }
    l += __shfl_xor(l, 32);

    // O = O^T / l: register r of block b is dim 32 b + 8 (r / 4) + 4 h + r % 4 of query qrow
    if (qrow < S) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        uint16_t* op = a.o + (int64_t)qrow * a.ldo + head * kD;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d = 32 * b + 8 * g + 4 * h;
                *reinterpret_cast<uint2*>(op + d) = uint2{pack_bf16(oacc[b][4 * g] * inv, oacc[b][4 * g + 1] * inv),
                                                          pack_bf16(oacc[b][4 * g + 2] * inv, oacc[b][4 * g + 3] * inv)};
            }
    }
}

}  // namespace

hipError_t launch_sdpa_prefill(const uint16_t* q, int64_t ldq, const uint16_t* k, int64_t ldk, const uint16_t* v,
                               int64_t ldv, uint16_t* o, int64_t ldo, int S, int H, int H_KV, uint16_t* k_cache,
                               uint16_t* v_cache, int cap, hipStream_t stream) {
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&sdpa_prefill_kernel),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (attr != hipSuccess) return attr;
    PrefillArgs a{};
    a.q = q;
    a.k = k;
    a.v = v;
    a.o = o;
    a.ldq = ldq;
    a.ldk = ldk;
    a.ldv = ldv;
    a.ldo = ldo;
    a.S = S;
    a.H = H;
    a.H_KV = H_KV;
    a.qtiles = (S + kBQ - 1) / kBQ;
    a.nslot = device_info().num_cu;
    a.scale2 = 1.4426950408889634f / sqrtf((float)kD);
    a.lazy = kLazy / a.scale2;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.cap = cap;
    hipLaunchKernelGGL(sdpa_prefill_kernel, dim3(a.qtiles * H), dim3(256), kLds, stream, a);
    return hipGetLastError();
}

}  // namespace nmi
