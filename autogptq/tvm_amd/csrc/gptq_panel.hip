// PANEL kernel: the product on the tiled format (gptq_tiled.hip) for long prompts and training batches, and the transposed
// product for the gradient, for any number of rows.
//
// A workgroup owns 32 RT rows x 256 columns.  x comes to LDS in blocks of 64 positions, straight from the row-major matrix and
// without passing through registers, and serves all waves; a wave owns 64 of the columns, keeps its 32 RT x 64 result in the
// accumulation registers and forms its weights in registers exactly once per workgroup, as the reference rounds them
// (fp16(scale * (q - zero))).  The words and (scale, zero) entries ride through LDS as well, so that every request of the walk
// is a copy into LDS that the wave counts itself; they run a block further ahead than x, because their dequantisation is
// spread between the matrix instructions of the step before.
//
// What bounds it (MI355X, 4096 rows on 8192 x 28672 int4, RT = 8): the chip's power.
// It runs at 1.56 of 2.4 GHz with the matrix pipes busy in 71 % of the cycles.  Matrix instructions alone sustain 1950 to 1990
// TFLOP/s in the 16 x 16 x 32 shape and 1700 to 1750 in the 32 x 32 x 16 one (which reads and writes each result twice as often
// per product), hence the former; on zeros, at full clock, both 2430 to 2460.  The kernel reaches 1320 to 1400, the dense library
// product of that size 1210.  Taking out the requests of the walk or the dequantisation gives back 15 to 18 % and 13 % of the time
// (RT = 4: 19 % and 16 %; three bits at RT = 5: 10 % and 26 %).
// The matmul kernel of gptq_tiled.hip, whose workgroups share nothing, takes 2000 us for what takes 1410 here.
// Below that, instruction issue: a wave alone on its SIMD issues an instruction per 5 clocks, so that two fit behind a
// 16-clock matrix instruction.  RT = 8 has 2.3 of them per matrix instruction, RT = 4 has 3.7: up to four row tiles two
// groups of four waves therefore take every other block each (two waves per SIMD, 256 registers each) and add up at the end.
// (Eight waves that split the rows instead would all form the same weights: 1500 us against 1385.)
// Deeper prefetching changed nothing (six stages against three at RT = 4: 67.9 us and 66.5).
#include "gptq_tiled_common.h"

namespace gptq {

struct PanelTail {
    const void *bias;        // fp16 [N] or nullptr
    void *y;                 // fp16 [M, N]
    float *partial;          // [split_k][rows of the tail][N] when split_k > 1
    const int32_t *out_map;  // TRANS: channel of result column p (nullptr = identity)
    uint32_t q_bytes, s_bytes;
    int col_wgs, main_rbs, tail_rbs, split_k, tail_steps, lb_per_group, G;
    // what the divisors of the first addresses are multiplied by instead (panel_div)
    uint32_t column_group_magic, tail_magic, lb_magic, tile_magic;
    uint32_t step_groups, step_rem;   // 2 x wave groups of lane blocks: whole groups, and the rest
};

// n / d by one multiplication, magic = floor(2^32 / d) + 1: exact while n d < 2^32 (e = d magic - 2^32 <= d adds less than 1 / d).
// 0 stands for d = 1; the host takes 1 for sizes beyond, which are divided.
static uint32_t panel_magic(unsigned long long most, uint32_t d)
{
    return d <= 1 ? 0u : (most * d < (1ull << 32) ? (uint32_t)((1ull << 32) / d) + 1u : 1u);
}
__device__ __forceinline__ uint32_t panel_div(uint32_t n, uint32_t d, uint32_t magic)
{
    if (magic == 1u) return n / d;
    return magic ? __umulhi(n, magic) : n;
}

// A request brings 1 KB (or 256 bytes) from a buffer into LDS: lane i's 16 (4) bytes land at lds + off + 16 i (4 i).  Inline
// assembly, so that the compiler does not wait for every outstanding request before each read of LDS; the kernel counts
// its requests itself.  LDS address and request want an instruction between them: a matrix instruction where one is due.
#define GPTQ_DMA(SIZE, BETWEEN, ...)                                                                                       \
    asm volatile("s_add_u32 m0, %[lds], %[off]\n\t" BETWEEN "\n\tbuffer_load_" SIZE " %[v], %[r], %[so] offen lds" __VA_ARGS__ \
                 [lds] "s"(lds), [off] "i"(off), [v] "v"(voff), [r] "s"(rsrc), [so] "s"(soff)                               \
                 : "scc")
template <int BYTES>
__device__ __forceinline__ void panel_request(uint32_t lds, int off, uint32_t voff, u4 rsrc, uint32_t soff)
{
    if constexpr (BYTES == 16) GPTQ_DMA("dwordx4", "s_nop 0", ::);
    if constexpr (BYTES == 12) GPTQ_DMA("dwordx3", "s_nop 0", ::);
    if constexpr (BYTES == 4) GPTQ_DMA("dword", "s_nop 0", ::);
}
// acc += b (16 columns) x a (16 rows), 32 positions.  Assembly, because it keeps the result in the accumulation registers:
// through the builtin the compiler moved half of them back and forth on every step.
__device__ __forceinline__ void panel_mfma(f4 &acc, u4 b, h8 a)
{
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}
__device__ __forceinline__ void panel_pin(f4 &acc) { asm volatile("" : "+a"(acc)); }
template <int BYTES>
__device__ __forceinline__ void panel_mfma_request(f4 &acc, u4 b, h8 a, uint32_t lds, int off, uint32_t voff, u4 rsrc, uint32_t soff)
{
#define GPTQ_MFMA "v_mfma_f32_16x16x32_f16 %[c], %[b], %[a], %[c]"
    if constexpr (BYTES == 16) GPTQ_DMA("dwordx4", GPTQ_MFMA, : [c] "+a"(acc) : [b] "v"(b), [a] "v"(a),);
    if constexpr (BYTES == 12) GPTQ_DMA("dwordx3", GPTQ_MFMA, : [c] "+a"(acc) : [b] "v"(b), [a] "v"(a),);
    if constexpr (BYTES == 4) GPTQ_DMA("dword", GPTQ_MFMA, : [c] "+a"(acc) : [b] "v"(b), [a] "v"(a),);
#undef GPTQ_MFMA
}
#undef GPTQ_DMA

__device__ __forceinline__ u4 buffer_of(const void *base, uint32_t bytes)
{
    const uint64_t a = (uint64_t)base;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32));
    return (u4){lo, hi & 0xffffu, (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}

template <int N>
__device__ __forceinline__ void wait_and_meet()
{
    // this wave's requests but for the last N have arrived, its LDS reads are done; then every wave's are
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// The unpack of this kernel.  The matrix instruction takes 32 positions in four octets, one per 16 lanes; lane (i, q) of step
// t (0, 1) takes octet 4 (q / 2) + 2 (q % 2) + t of a block of 64, i.e. operand j = 2 (q % 2) + t of the tiled format's lane
// slot (column, q / 2).  read() brings the words that both steps of a lane need; operand() is TileCodec's unpack of
// operand j with j's lane part folded into the address (2, 4, 8 bits) or into selected words and shifts (3 bits).
template <int BITS>
struct PanelCodec {
    static constexpr int WORDS = BITS == 2 ? 1 : (BITS == 4 ? 2 : 4);
    // byte offset, inside a tile's place in LDS, of what lane slot (column n of 32, half h) reads for the pair of operands p
    static __device__ uint32_t at(uint32_t n, uint32_t h, uint32_t p)
    {
        const uint32_t slot = h * 32u + n;
        if (BITS == 2) return slot * 8u + p * 4u;
        if (BITS == 4) return slot * 16u + p * 8u;
        if (BITS == 8) return slot * 16u + p * 1024u;
        return slot * 16u + p * 4u;   // (three words take the place of four)
    }
    // odd: the lanes of pair 1 (operands 2, 3)
    static __device__ __forceinline__ u4 read(const char *src, bool odd)
    {
        if constexpr (BITS == 2) {
            return (u4){*(const uint32_t *)src, 0u, 0u, 0u};
        } else if constexpr (BITS == 4) {
            const u2 v = *(const u2 *)src;
            return (u4){v[0], v[1], 0u, 0u};
        } else if constexpr (BITS == 8) {
            return *(const u4 *)src;
        } else {
            // The windows of the two operands (biased3_block keeps bits 0..5 and 18..23 of each) from words (0, 1) or (1, 2):
            //   pair 0: w1:w0, w1:w0 >> 6, w1:w0 >> 12, w1 >> 4;   pair 1: w2:w1 >> 10, w2:w1 >> 16, w2 >> 8, w2 >> 14 | w2 >> 2
            const uint32_t lo = *(const uint32_t *)src, hi = *(const uint32_t *)(src + 4);
            const uint32_t x = hi >> (odd ? 14u : 4u), y = hi >> (odd ? 2u : 4u);
            return (u4){__builtin_amdgcn_alignbit(hi, lo, odd ? 10u : 0u), __builtin_amdgcn_alignbit(hi, lo, odd ? 16u : 6u),
                        __builtin_amdgcn_alignbit(hi, odd ? hi : lo, odd ? 8u : 12u), (x & 0xffffu) | (y & 0xffff0000u)};
        }
    }
    // register r (two positions: base + code) of the operand of step t
    static __device__ __forceinline__ uint32_t pair(const u4 &w, int t, int r, const uint32_t (&mg)[TileCodec<BITS>::KINDS])
    {
        if constexpr (BITS == 2) {
            const uint32_t v = t ? w[0] >> 8 : w[0];
            return and_or(v, 0x00030003u << (2 * r), mg[r]);
        } else if constexpr (BITS == 4) {
            const uint32_t v = r < 2 ? w[t] : w[t] >> 8;
            return and_or(v, r & 1 ? 0x00f000f0u : 0x000f000fu, mg[r & 1]);
        } else if constexpr (BITS == 8) {
            const uint32_t v = r & 1 ? w[2 * t + r / 2] >> 8 : w[2 * t + r / 2];
            return and_or(v, 0x00ff00ffu, mg[0]);
        } else {
            return and_or(w[2 * t + r / 2], r & 1 ? 0x00e00038u : 0x001c0007u, mg[r & 1]);
        }
    }
};

// pieces (of sixteen) begun before matrix instruction i of `all`, the first behind instruction `first`, the last early enough
// that its second part has an instruction to follow
constexpr int panel_pieces(int i, int all, int first)
{
    const int fit = (all - 2 - first) * 16 / 15, span = fit < all ? fit : all, k = (16 * (i - first) + span - 1) / span;
    return i <= first ? 0 : (k < 16 ? k : 16);
}

template <int BITS, int RT, bool TRANS>
__global__ __launch_bounds__(256 * panel_waves_k(RT)) void panel_kernel(const _Float16 *x, const char *qtile, const uint32_t *sz, int M, int ldx,
                                                       int N, int S_total, int T_total, const PanelTail t)
{
    using Codec = TileCodec<BITS>;
    constexpr int KINDS = Codec::KINDS;
    constexpr int CT = 2, NW = 4;
    constexpr int BW = 256 * BITS;                       // bytes of one tile's block
    constexpr int NB = BITS == 8 || BITS == 2 ? 2 : 1;   // requests per block
    constexpr int NLB = CT * NB + CT, NL = RT + NLB;     // requests per wave and step: words and scales; and x
    constexpr int BL = panel_tile_bytes(BITS);           // a tile's place in LDS
    constexpr int B_OFF = RT * 4096, S_OFF = B_OFF + NW * CT * BL;
    constexpr int KW = panel_waves_k(RT);                // wave groups: block s KW + kw of the walk belongs to group kw
    constexpr uint32_t PART = panel_block_bytes(BITS, RT), STAGE = KW * PART;
    constexpr int STAGES = panel_stages(BITS, RT);
    // A step (a block of 64) is GROUPS groups of four matrix instructions that share a fragment of x; fragments are read
    // RING groups ahead.  The waves meet at group MEET: LATE groups after the last read of the block, so that the reads
    // have come back by then; the reads of the next block's first fragments catch up there.
    constexpr int MT = 2 * RT, NC = 2 * CT, GROUPS = 2 * MT;
    constexpr int RING = RT == 1 ? 2 : (RT < 4 ? 4 : (RT % 2 ? RT : (RT == 6 ? 6 : 8)));
    constexpr int MEET = GROUPS - RING + (RT == 1 ? 1 : 2);
    static_assert(MEET > MT && GROUPS % RING == 0);

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = w / NW, nw = w % NW;
    const int i16 = lane & 15, q4 = lane >> 4;

    // The first main_rbs row blocks take all of K each, the tail_rbs after them K in split_k ranges: whole turns of the chip,
    // and what is left of the rows spread over one turn more.
    // XCD-aware order: workgroups are dealt to the XCDs round robin, so id % 8 names the XCD; each takes a
    // contiguous run of the tile order, in which groups of four row blocks walk the columns together
    int rb, cb, split = 0;
    const int n_main = t.col_wgs * t.main_rbs;
    const bool tail_wg = (int)blockIdx.x >= n_main;
    const bool ranges = tail_wg && t.split_k > 1;
    {
        const uint32_t row_wgs = tail_wg ? t.tail_rbs : t.main_rbs, nwg = t.col_wgs * row_wgs;
        uint32_t id = blockIdx.x - (tail_wg ? n_main : 0);
        if (ranges) split = (int)panel_div(id, nwg, t.tail_magic), id -= split * nwg;
        const uint32_t q = nwg / 8, r = nwg % 8, xcd = id % 8, i = id / 8;
        const uint32_t lin = xcd * q + min(xcd, r) + i;
        const uint32_t per = 4 * t.col_wgs, grp = panel_div(lin, per, t.column_group_magic), in = lin - grp * per;
        const uint32_t rows = min(4u, row_wgs - 4 * grp);
        const uint32_t c = rows == 4 ? in / 4 : (rows == 3 ? in / 3 : (rows == 2 ? in / 2 : in));
        cb = (int)c;
        rb = (int)(4 * grp + (in - c * rows)) + (tail_wg ? t.main_rbs : 0);
    }
    const int wg_steps = tail_wg ? t.tail_steps : S_total;
    const int row0 = rb * 32 * RT;
    const int T0 = cb * NW * CT + nw * CT;
    const int S_begin = split * wg_steps, S_last = S_total - 1;
    const int S_end = min(S_begin + wg_steps, S_total), steps = (S_end - S_begin + KW - 1) / KW;

    const u4 xr = buffer_of(x + (size_t)row0 * ldx, (uint32_t)min(M - row0, 32 * RT) * (uint32_t)ldx * 2u);
    const u4 qr = buffer_of(qtile, t.q_bytes);
    const u4 sr = buffer_of(sz, t.s_bytes);

    // x: request i of this wave brings rows 8 (nw RT + i) .. + 7 of the block, 128 bytes each (rows past M lie outside the
    // buffer and read as zeros).  LDS keeps a row's eight 16-byte octets at octet ^ f(row), f = (row & 7) ^ ((row >> 3) & 1):
    // the reads of a fragment (16 rows x 4 octets) then spread over all banks.  The second wave group swaps the halves of a row
    // tile (16 rows each): see the result.
    uint32_t xo[RT];
#pragma unroll
    for (int i = 0; i < RT; i++) {
        const int blk = nw * RT + i;
        const int oct = (lane & 7) ^ (lane >> 3) ^ (blk & 1);
        xo[i] = (uint32_t)(8 * (blk ^ (2 * kw)) + (lane >> 3)) * (uint32_t)ldx * 2u + (uint32_t)oct * 16u;
    }
    // a block past the workgroup's range (a walk of an odd count of blocks), and the half of a last block that lies past K,
    // are sent out of the buffer's range as well
    const uint32_t tail = ((uint32_t)lane ^ (uint32_t)(lane >> 3)) & 4u ? 0x80000000u : 0u;
    const int S_cut = ldx % 64 != 0 && S_end == S_total ? S_last : S_end;
    auto cut = [&](int S) {
        if (S >= S_cut) {
            asm volatile("");   // (once per wave: not worth a select per request)
            const uint32_t bits = S < S_end ? tail : 0x80000000u;
#pragma unroll
            for (int i = 0; i < RT; i++) xo[i] |= bits;
        }
    };

    uint32_t q_base[CT], s_base[CT];
#pragma unroll
    for (int i = 0; i < CT; i++) {
        const int T = min(T0 + i, T_total - 1);   // (a missing tile repeats the last one; it is never stored)
        q_base[i] = (uint32_t)T * (uint32_t)S_total * (uint32_t)BW;
        s_base[i] = TRANS ? panel_div((uint32_t)T, (uint32_t)t.lb_per_group, t.tile_magic) * (uint32_t)S_total * 256u : 128u * (uint32_t)T;
    }
    // the group of this lane's half of the block requested next, as an offset into sz; a step moves on by 2 KW runs of 32 positions
    const uint32_t row_bytes = 4u * (uint32_t)N, lbg = (uint32_t)t.lb_per_group;
    const uint32_t lb0 = 2u * (uint32_t)(S_begin + kw) + (uint32_t)(lane >> 5);
    const uint32_t g0 = panel_div(lb0, lbg, t.lb_magic);
    uint32_t g_off = g0 * row_bytes + (uint32_t)(lane & 31) * 4u, g_rem = lb0 - g0 * lbg;
    const uint32_t g_skip = t.step_groups * row_bytes, g_inc = t.step_rem;
    auto next_group = [&]() {
        g_rem += g_inc;
        const bool over = g_rem >= lbg;
        g_off += g_skip + (over ? row_bytes : 0u);
        g_rem -= over ? lbg : 0u;
    };
    const uint32_t part = (uint32_t)kw * PART;
    const uint32_t a_dst = part + (uint32_t)nw * (RT * 1024u), b_dst = part + B_OFF + (uint32_t)(nw * CT * BL), s_dst = part + S_OFF + (uint32_t)(nw * CT * 256);
    const uint32_t l_words = lane * (BITS == 2 ? 4u : (BITS == 3 ? 12u : 16u));
    // A block past the range brings no scales either: zeros times its weights have to be zero, and they are not where a weight
    // is infinite.
    uint32_t t_off = lane * 4u;
    auto cut_scales = [&](int S) {
        if (S >= S_end) {
            asm volatile("");
            (TRANS ? t_off : g_off) |= 0x80000000u;
        }
    };

    // request d of a step: x of block Sa to the stage at byte `sa`, words and scales of block Sb to the one at `sb`
    auto request = [&](auto d_c, uint32_t sa, int Sa, uint32_t sb, int Sb, auto &&go) {
        constexpr int d = decltype(d_c)::value;
        if constexpr (d < CT * NB) {
            constexpr int i = d / NB, e = d % NB;
            constexpr int bytes = BITS == 2 ? 4 : (BITS == 3 ? 12 : 16);
            go(std::integral_constant<int, bytes>{}, sb + b_dst, i * BL + e * bytes * 64, l_words, qr,
               q_base[i] + (uint32_t)Sb * (uint32_t)BW + e * (bytes * 64));
        } else if constexpr (d < NLB) {
            constexpr int i = d - CT * NB;
            go(std::integral_constant<int, 4>{}, sb + s_dst, i * 256, TRANS ? t_off : g_off, sr,
               TRANS ? s_base[i] + (uint32_t)Sb * 256u : s_base[i]);
        } else {
            constexpr int i = d - NLB;
            go(std::integral_constant<int, 16>{}, sa + a_dst, i * 1024, xo[i], xr, (uint32_t)Sa * 128u);
        }
    };
    auto request_now = [&](auto from_c, auto n_c, uint32_t sa, int Sa, uint32_t sb, int Sb) {
        constexpr int from = decltype(from_c)::value;
        [&]<int... D>(std::integer_sequence<int, D...>) {
            (request(std::integral_constant<int, from + D>{}, sa, Sa, sb, Sb,
                     [](auto bytes_c, uint32_t lds, int off, uint32_t v, u4 r, uint32_t so) {
                         panel_request<decltype(bytes_c)::value>(lds, off, v, r, so);
                     }), ...);
        }(std::make_integer_sequence<int, decltype(n_c)::value>{});
    };

    // the result in tiles of 16 columns x 16 rows: element v of lane (i, q) of tile (mt, c) is row 16 mt + i, column
    // 16 c + 4 q + v
    f4 acc[MT][NC];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[mt][c] = (f4){0.f, 0.f, 0.f, 0.f};

    // words and scales run one block further ahead than x: they are in registers a step before they are used
    const int S_wave = S_begin + kw;
    cut_scales(S_wave);
    request_now(std::integral_constant<int, 0>{}, std::integral_constant<int, NLB>{}, 0, 0, 0, min(S_wave, S_last));
#pragma unroll
    for (int u = 0; u < STAGES - 1; u++) {
        next_group();
        cut(S_wave + KW * u);
        cut_scales(S_wave + KW * (u + 1));
        request_now(std::integral_constant<int, 0>{}, std::integral_constant<int, NL>{}, u * STAGE, min(S_wave + KW * u, S_last),
                    (u + 1) * STAGE, min(S_wave + KW * (u + 1), S_last));
    }

    uint32_t mg[KINDS];
    tile_magic<BITS>(mg);
    // where the fragment of row tile mt and step t lies in a stage: + 2048 mt; words and scales (u: 16-column half of a tile)
    uint32_t a_at[2], b_at[2], s_at[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
        const int oct = 4 * (q4 >> 1) + 2 * (q4 & 1) + u;
        a_at[u] = part + (uint32_t)i16 * 128u + (uint32_t)((oct ^ (i16 & 7) ^ (i16 >> 3)) * 16);
        b_at[u] = b_dst + PanelCodec<BITS>::at(16 * u + i16, q4 >> 1, q4 & 1);
        s_at[u] = s_dst + (TRANS ? (uint32_t)oct * 32u : (uint32_t)(32 * (q4 >> 1) + 16 * u + i16) * 4u);
    }
    const bool odd = q4 & 1;

    u4 wd[NC];
    uint32_t sn[NC];
    u4 tq[2][CT][2];
    h2 cs[NC], czb[NC][KINDS];
    u4 b[2][NC];
    h8 a[RING];
    auto read_a = [&](uint32_t st, int g) { return *(const h8 *)(smem + (st + a_at[g / MT] + (g % MT) * 2048)); };
    // part c of a block's words and scales
    auto read_words = [&](uint32_t st, int c) {
        wd[c] = PanelCodec<BITS>::read((const char *)smem + (st + b_at[c & 1] + (c >> 1) * BL), odd);
        if constexpr (TRANS) {
            tq[c & 1][c >> 1][0] = *(const u4 *)(smem + (st + s_at[c & 1] + (c >> 1) * 256));
            tq[c & 1][c >> 1][1] = *(const u4 *)(smem + (st + s_at[c & 1] + (c >> 1) * 256 + 16));
        } else {
            sn[c] = *(const uint32_t *)(smem + (st + s_at[c & 1] + (c >> 1) * 256));
        }
    };
    // piece k (0..15) of the operands of step t: register k % 4 of column tile k / 4, exactly as the reference rounds it
    // ((base + q) - (base + zero) is exact, the product rounds once); in two parts, for the product waits for the difference
    h2 diff[16];
    auto subtract = [&](auto k_c, auto t_c) {
        constexpr int k = decltype(k_c)::value, t = decltype(t_c)::value, c = k / 4, r = k % 4;
        if constexpr (!TRANS && t == 0 && r == 0) {
            const h2 v = as_h2(sn[c]);
            cs[c] = (h2){v[0], v[0]};
#pragma unroll
            for (int e = 0; e < KINDS; e++)
                czb[c][e] = (h2){v[1], v[1]} + (h2){(_Float16)Codec::base(2 * e), (_Float16)Codec::base(2 * e + 1)};
        }
        const h2 v = as_h2(PanelCodec<BITS>::pair(wd[c], t, r, mg));
        diff[k] = v - (TRANS ? as_h2(tq[t][c >> 1][1][r]) : czb[c][r % KINDS]);
    };
    auto scale = [&](auto k_c, auto t_c) {
        constexpr int k = decltype(k_c)::value, t = decltype(t_c)::value, c = k / 4, r = k % 4;
        b[t][c][r] = as_u32(diff[k] * (TRANS ? as_h2(tq[t][c >> 1][0][r]) : cs[c]));
    };

    wait_and_meet<(STAGES - 2) * NL>();
#pragma unroll
    for (int c = 0; c < NC; c++) read_words(0, c);
    [&]<int... P>(std::integer_sequence<int, P...>) {
        (subtract(std::integral_constant<int, P>{}, std::integral_constant<int, 0>{}), ...);
        (scale(std::integral_constant<int, P>{}, std::integral_constant<int, 0>{}), ...);
    }(std::make_integer_sequence<int, 16>{});
#pragma unroll
    for (int g = 0; g < RING; g++) a[g] = read_a(0, g);
    __builtin_amdgcn_sched_barrier(0);

    // Between two matrix instructions (16 clocks each) a wave can issue three others, so that each has its share of them
    // behind it: of a group's four, the first a request, the second the differences of a piece, the third its products,
    // the fourth a read.
    uint32_t cur = 0, nxt = STAGE, far = (STAGES - 1) * STAGE;   // stages of blocks s, s + 1, s + STAGES - 1
    uint32_t nxt2 = 0, far2 = 0;
    int Su = S_wave + KW * (STAGES - 1);   // the block requested in this step (words and scales: KW further)
    int Sa = min(Su, S_last), Sb = min(Su + KW, S_last);
    for (int s = 0; s < steps; s++) {
        [&]<int... I>(std::integer_sequence<int, I...>) {
            ([&] {
                constexpr int m = I, g = m / NC, c = m % NC, t = g / MT, mt = g % MT;
                if constexpr (m == 0) {
                    next_group();
                } else if constexpr (m == 1) {
                    cut(Su);
                } else if constexpr (m == 2) {
                    cut_scales(Su + KW);
                }
                if constexpr (m == MEET * NC) wait_and_meet<(STAGES - 2) * NL>();   // x of the next block is in LDS, this one's has been read
                constexpr int d0 = g * NL / MEET, d1 = (g + 1) * NL / MEET;
                if constexpr (g < MEET && c == 0 && d1 > d0) {
                    request(std::integral_constant<int, d0>{}, far, Sa, cur, Sb,
                            [&](auto bytes_c, uint32_t lds, int off, uint32_t v, u4 r, uint32_t so) {
                                panel_mfma_request<decltype(bytes_c)::value>(acc[mt][c], b[t][c], a[g % RING], lds, off, v, r, so);
                            });
                    request_now(std::integral_constant<int, d0 + 1>{}, std::integral_constant<int, d1 - d0 - 1>{}, far, Sa, cur, Sb);
                } else {
                    panel_mfma(acc[mt][c], b[t][c], a[g % RING]);
                }
                // words and scales of the next block at the head of the second step
                if constexpr (t == 1 && mt == 0) read_words(nxt, c);
                if constexpr (c == NC - 1) {
                    if constexpr (g + RING < GROUPS) {
                        a[g % RING] = read_a(cur, g + RING);
                    } else if constexpr (g == MEET) {
#pragma unroll
                        for (int e = GROUPS - RING; e <= g; e++) a[e % RING] = read_a(nxt, e + RING - GROUPS);
                    } else if constexpr (g > MEET) {
                        a[g % RING] = read_a(nxt, g + RING - GROUPS);
                    }
                }
                // pieces: the operands of this block's second step in its first, the next block's first ones in its second,
                // from the third group on (the words have come by then)
                constexpr int ph = m - t * MT * NC, first = t == 0 ? 1 : (MT > 2 ? 2 * NC + 1 : NC);
                constexpr int pp = panel_pieces(ph - 1, MT * NC, first), p0 = panel_pieces(ph, MT * NC, first),
                              p1 = panel_pieces(ph + 1, MT * NC, first);
                [&]<int... P>(std::integer_sequence<int, P...>) {
                    (scale(std::integral_constant<int, pp + P>{}, std::integral_constant<int, 1 - t>{}), ...);
                }(std::make_integer_sequence<int, p0 - pp>{});
                [&]<int... P>(std::integer_sequence<int, P...>) {
                    (subtract(std::integral_constant<int, p0 + P>{}, std::integral_constant<int, 1 - t>{}), ...);
                }(std::make_integer_sequence<int, p1 - p0>{});
                // the next step's blocks and stages, once the requests are out
                if constexpr (m == MEET * NC + 1) {
                    Su += KW, Sa = min(Su, S_last), Sb = min(Su + KW, S_last);
                } else if constexpr (m == MEET * NC + 2) {
                    nxt2 = nxt + STAGE == STAGES * STAGE ? 0 : nxt + STAGE;
                    far2 = far + STAGE == STAGES * STAGE ? 0 : far + STAGE;
                }
                __builtin_amdgcn_sched_barrier(0);
            }(), ...);
        }(std::make_integer_sequence<int, GROUPS * NC>{});
        cur = nxt, nxt = nxt2, far = far2;
    }

    // ---- the result ----
    // (the compiler does not know of the matrix instructions in flight: their results want 18 cycles)
    asm volatile("s_nop 15\n\ts_nop 7\n\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // In pieces of 16 rows x 64 columns, RT of them per wave: two wave groups add up in LDS, each wave hands over every other
    // piece (acc[2 rt + 1]; the second group holds the halves of a row tile the other way round, so that it keeps what the first hands
    // over); a group alone finishes all 2 RT.  A finished piece is turned around in LDS of the wave's own and stored
    // in rows.  (One exchange, the same code for both groups and each with half of the work, where the groups took turns at whole row
    // tiles, an exchange per two of them: 333 rows of 5120 x 3424 int8 27.5 -> 27.0 us, 701 of 7936 x 1600 33.8 -> 33.0, 1000 of 8192 x 8192
    // 113.4 -> 111.8; a quarter of a row per four lanes, stored without turning the piece, was slower than before.)
    constexpr int SLOT = 4096;
    unsigned char *give = smem + w * (RT * SLOT), *take = KW == 2 ? smem + (w ^ NW) * (RT * SLOT) : smem + w * (4 * SLOT);
    const int c8 = (lane & 7) * 8, T8 = T0 + (c8 >> 5);
    f4 bias[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        bias[c] = (f4){0.f, 0.f, 0.f, 0.f};
        if (!TRANS && t.bias && !ranges) {
            const h4 v = *(const h4 *)((const _Float16 *)t.bias + 32 * min(T0 + (c >> 1), T_total - 1) + 16 * (c & 1) + 4 * q4);
            bias[c] = (f4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
        }
    }
    int to[8];
    if (TRANS && t.out_map) {
        const int p0 = 32 * min(T8, T_total - 1) + (c8 & 31);
        const int4 u = *(const int4 *)(t.out_map + p0), v = *(const int4 *)(t.out_map + p0 + 4);
        to[0] = u.x, to[1] = u.y, to[2] = u.z, to[3] = u.w, to[4] = v.x, to[5] = v.y, to[6] = v.z, to[7] = v.w;
#pragma unroll
        for (int e = 0; e < 8; e++) to[e] = min(max(to[e], 0), N - 1);
    }
    _Float16 *y = (_Float16 *)t.y;
    if constexpr (KW == 2) {
#pragma unroll
        for (int rt = 0; rt < RT; rt++)
#pragma unroll
            for (int c = 0; c < NC; c++) *(f4 *)(give + rt * SLOT + c * 1024 + lane * 16) = acc[2 * rt + 1][c];
        __syncthreads();
    }
    // two pieces at a time: rows row0 + 16 mt .. + 15 (the second group's, 16 further on)
    constexpr int PIECES = KW == 2 ? RT : 2 * RT;
    [&]<int... I>(std::integer_sequence<int, I...>) {
        ([&] {
            constexpr int n = 2 * I + 1 < PIECES ? 2 : 1;
            unsigned char *slot[2];
            f4 sum[2][NC];
            int first[2];
#pragma unroll
            for (int e = 0; e < n; e++) {
                const int mt = KW == 2 ? 2 * (2 * I + e) : 2 * I + e;
                slot[e] = take + (KW == 2 ? 2 * I + e : (2 * I + e) % 4) * SLOT;
                first[e] = row0 + 16 * mt + (KW == 2 ? 16 * kw : 0);
#pragma unroll
                for (int c = 0; c < NC; c++) panel_pin(acc[mt][c]);   // (the others stay in the accumulation registers until their turn)
#pragma unroll
                for (int c = 0; c < NC; c++)
                    sum[e][c] = acc[mt][c] + (KW == 2 ? *(const f4 *)(slot[e] + c * 1024 + lane * 16) + bias[c] : bias[c]);
            }
            if (ranges) {
                // (16 bytes of a row at place ^ row)
                const int tail0 = 32 * RT * t.main_rbs;
                const int c4 = (lane & 15) * 4, T4 = T0 + (c4 >> 5);
#pragma unroll
                for (int e = 0; e < n; e++)
#pragma unroll
                    for (int c = 0; c < NC; c++) *(f4 *)(slot[e] + i16 * 256 + ((4 * c + q4) ^ i16) * 16) = sum[e][c];
#pragma unroll
                for (int e = 0; e < n; e++)
#pragma unroll
                    for (int it = 0; it < 4; it++) {
                        const int m = 4 * it + (lane >> 4), row = first[e] + m;
                        const f4 v = *(const f4 *)(slot[e] + m * 256 + ((lane & 15) ^ m) * 16);
                        if (row < M && T4 < T_total) *(f4 *)(t.partial + ((size_t)split * (M - tail0) + (row - tail0)) * (size_t)N + 32 * T4 + (c4 & 31)) = v;
                    }
            } else {
#pragma unroll
                for (int e = 0; e < n; e++)
#pragma unroll
                    for (int c = 0; c < NC; c++) {
                        h4 o;
#pragma unroll
                        for (int v = 0; v < 4; v++) o[v] = (_Float16)sum[e][c][v];
                        *(h4 *)(slot[e] + i16 * 144 + (16 * c + 4 * q4) * 2) = o;
                    }
#pragma unroll
                for (int e = 0; e < n; e++)
#pragma unroll
                    for (int it = 0; it < 2; it++) {
                        const int m = 8 * it + (lane >> 3), row = first[e] + m;
                        const h8 v = *(const h8 *)(slot[e] + m * 144 + c8 * 2);
                        if (row < M && T8 < T_total) {
                            if (TRANS && t.out_map) {
#pragma unroll
                                for (int k = 0; k < 8; k++) y[(size_t)row * N + to[k]] = v[k];
                            } else {
                                *(h8 *)(y + (size_t)row * N + 32 * T8 + (c8 & 31)) = v;
                            }
                        }
                    }
            }
            __builtin_amdgcn_sched_barrier(0);
        }(), ...);
    }(std::make_integer_sequence<int, (PIECES + 1) / 2>{});
}

// xs[m][p] = x[m][xsrc[p]]: the activations in the order of the tiled copy.  A workgroup takes ROWS rows and one of gridDim.y
// parts of K: the rows go to LDS with coalesced loads, the gather reads LDS, and the index vectors are read once for all of
// them (2048 x 4096: 7.4 to 9.8 us for 33 MB of traffic; a pass that writes ready-made fragments took 21).
template <int ROWS>
__global__ __launch_bounds__(256) void panel_gather_kernel(const _Float16 *__restrict__ x, const int32_t *__restrict__ xsrc,
                                                           _Float16 *__restrict__ xs, int M, int K)
{
    const int row0 = blockIdx.x * ROWS, rows = min(ROWS, M - row0);
    _Float16 *xl = (_Float16 *)smem;
    const u4 *src = (const u4 *)(x + (size_t)row0 * K);
    // the first index vectors, and four requests of x at a time: one after the other they are a chain of latencies
    const int o0 = blockIdx.y * 256 + threadIdx.x, oc = min(o0, K / 8 - 1), all = rows * (K / 8);
    int4 u = *(const int4 *)(xsrc + 8 * oc), v = *(const int4 *)(xsrc + 8 * oc + 4);
    for (int i = threadIdx.x; i < all; i += 1024) {
        u4 q[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i + 256 * j < all) q[j] = src[i + 256 * j];
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i + 256 * j < all) ((u4 *)xl)[i + 256 * j] = q[j];
    }
    __syncthreads();
    for (int o = o0; o < K / 8; o += 256 * gridDim.y) {
        if (o > o0) u = *(const int4 *)(xsrc + 8 * o), v = *(const int4 *)(xsrc + 8 * o + 4);
        int idx[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; e++) idx[e] = min(max(idx[e], 0), K - 1);   // a bad map must not fault
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            if (r >= rows) break;
            h8 out;
#pragma unroll
            for (int e = 0; e < 8; e++) out[e] = xl[r * K + idx[e]];
            *(h8 *)(xs + (size_t)(row0 + r) * K + 8 * o) = out;
        }
    }
}

// The way back for the transposed product: gx[m][xsrc[p]] = gs[m][p], or, from row tail0 on, the sum of the K ranges' partial results.  A row is
// put in order in LDS and leaves it in one piece (2048 x 4096: 6.1 to 8.3 us; stores of two bytes from the product itself cost 31).
__global__ __launch_bounds__(256) void panel_scatter_kernel(const _Float16 *__restrict__ gs, const float *__restrict__ partial,
                                                            const int32_t *__restrict__ xsrc, _Float16 *__restrict__ gx, int M,
                                                            int K, int split, int tail0)
{
    const int row = blockIdx.x;
    _Float16 *xl = (_Float16 *)smem;
    for (int o = threadIdx.x; o < K / 8; o += 256) {
        const int4 u = *(const int4 *)(xsrc + 8 * o), v = *(const int4 *)(xsrc + 8 * o + 4);
        const int idx[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        h8 g;
        if (partial && row >= tail0) {
            f4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
            for (int s = 0; s < split; s++) {
                const f4 *p = (const f4 *)(partial + ((size_t)s * (M - tail0) + (row - tail0)) * K + 8 * o);
                a += p[0], b += p[1];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) g[e] = (_Float16)a[e], g[4 + e] = (_Float16)b[e];
        } else {
            g = *(const h8 *)(gs + (size_t)row * K + 8 * o);
        }
#pragma unroll
        for (int e = 0; e < 8; e++) xl[min(max(idx[e], 0), K - 1)] = g[e];
    }
    __syncthreads();
    u4 *dst = (u4 *)(gx + (size_t)row * K);
    for (int i = threadIdx.x; i < K / 8; i += 256) dst[i] = ((const u4 *)xl)[i];
}

template <typename Kern>
static bool allow_lds(Kern kern, int bytes)
{
    if (bytes <= 65536 || hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess)
        return true;
    (void)hipGetLastError();
    return false;
}

static int launch_panel_gather(const void *x, const int32_t *xsrc, void *xs, int M, int K, hipStream_t stream)
{
    auto go = [&](auto kern, int rows, int parts) {
        if (!allow_lds(kern, rows * K * 2)) return GPTQ_HIP_ERR_LAUNCH;
        hipLaunchKernelGGL(kern, dim3((M + rows - 1) / rows, parts), dim3(256), rows * K * 2, stream, (const _Float16 *)x, xsrc,
                           (_Float16 *)xs, M, K);
        return hipGetLastError() == hipSuccess ? GPTQ_HIP_OK : GPTQ_HIP_ERR_LAUNCH;
    };
    // several rows per workgroup once that leaves a few workgroups per CU; parts of a row while the rows are fewer than the CUs
    if (M >= 2048 && K <= 4096) return go(panel_gather_kernel<4>, 4, 1);
    if (M >= 1024 && K <= 16384) return go(panel_gather_kernel<2>, 2, 1);
    const int most = (K + 2047) / 2048, want = (kNumCUs + M - 1) / M;
    return go(panel_gather_kernel<1>, 1, want < most ? want : most);
}

static int launch_panel_scatter(const void *gs, const float *partial, const int32_t *xsrc, void *gx, int M, int K, int split,
                                int tail0, hipStream_t stream)
{
    if (!allow_lds(panel_scatter_kernel, K * 2)) return GPTQ_HIP_ERR_LAUNCH;
    hipLaunchKernelGGL(panel_scatter_kernel, dim3(M), dim3(256), K * 2, stream, (const _Float16 *)gs, partial, xsrc,
                       (_Float16 *)gx, M, K, split, tail0);
    return hipGetLastError() == hipSuccess ? GPTQ_HIP_OK : GPTQ_HIP_ERR_LAUNCH;
}

template <int BITS, int RT, bool TRANS>
static int launch_panel_one(const _Float16 *x, const char *qtile, const uint32_t *sz, int M, int ldx, int N, int S_total,
                            int T_total, const PanelTail &t, const gptq_hip_plan &plan, hipStream_t stream)
{
    auto kern = panel_kernel<BITS, RT, TRANS>;
    const int lds = panel_lds_bytes(BITS, RT);
    if (!allow_lds(kern, lds)) return GPTQ_HIP_ERR_LAUNCH;
    hipLaunchKernelGGL(kern, dim3((unsigned)t.col_wgs * ((unsigned)t.main_rbs + (unsigned)t.tail_rbs * (unsigned)t.split_k)), dim3(256 * panel_waves_k(RT)), lds,
                       stream, x, qtile, sz, M, ldx, N, S_total, T_total, t);
    return hipGetLastError() == hipSuccess ? GPTQ_HIP_OK : GPTQ_HIP_ERR_LAUNCH;
}

template <int BITS, bool TRANS>
static int launch_panel_bits(const _Float16 *x, const char *qtile, const uint32_t *sz, int M, int ldx, int N, int S_total,
                             int T_total, const PanelTail &t, const gptq_hip_plan &plan, hipStream_t stream)
{
    switch (plan.row_tiles) {
#define GPTQ_PANEL_CASE(R) \
    case R: return launch_panel_one<BITS, R, TRANS>(x, qtile, sz, M, ldx, N, S_total, T_total, t, plan, stream)
        GPTQ_PANEL_CASE(1);
        GPTQ_PANEL_CASE(2);
        GPTQ_PANEL_CASE(3);
        GPTQ_PANEL_CASE(4);
        GPTQ_PANEL_CASE(5);
        GPTQ_PANEL_CASE(6);
        GPTQ_PANEL_CASE(7);
        GPTQ_PANEL_CASE(8);
#undef GPTQ_PANEL_CASE
    }
    return GPTQ_HIP_ERR_UNSUPPORTED;
}

// y = x @ W (+ bias) on the tiled copy, or gx = gy @ W^T on its transposed form (trans): the reduction is K_red long,
// the result has N_out columns.
int launch_panel(const void *x, const void *qtile, const uint32_t *sz, const int32_t *xsrc, const void *bias, void *y,
                 void *xs, float *partial, int M, int K, int N, int bits, int group_size, bool trans, const gptq_hip_plan &plan,
                 void *stream_v)
{
    hipStream_t stream = (hipStream_t)stream_v;
    const int K_red = trans ? N : K, N_out = trans ? K : N;
    // Workgroups that with all their ranges are past the 2^32 threads of a launch: so many row blocks at a time (ranges along a second
    // dimension of the grid made every call of the kernel slower, 13 rows of 12640 x 30784 int3 51.6 -> 53.9 us, 1176 of 5120 x 3296 48.4 -> 49.1)
    const unsigned long long block_threads = (unsigned long long)plan.grid_x * plan.split_k * plan.block;
    const int most = (int)(((1ull << 32) - 1) / block_threads), block_rows = 32 * plan.row_tiles;
    if (plan.m_blocks > most && panel_main_blocks(plan) == 0) {
        for (int b = 0; b < plan.m_blocks; b += most) {
            gptq_hip_plan part = plan;
            part.m_blocks = part.grid_z = plan.m_blocks - b < most ? plan.m_blocks - b : most;
            const size_t row0 = (size_t)b * block_rows;
            const int rows = (int)((size_t)M - row0 < (size_t)most * block_rows ? M - row0 : (size_t)most * block_rows);
            const int rc = launch_panel((const _Float16 *)x + row0 * K_red, qtile, sz, xsrc, bias, (_Float16 *)y + row0 * N_out,
                                        xsrc ? (_Float16 *)xs + row0 * K : xs, partial, rows, K, N, bits, group_size, trans, part, stream_v);
            if (rc != GPTQ_HIP_OK) return rc;
        }
        return GPTQ_HIP_OK;
    }
    if (!trans && xsrc) {
        const int rc = launch_panel_gather(x, xsrc, xs, M, K, stream);
        if (rc != GPTQ_HIP_OK) return rc;
        x = xs;
    }
    const int S_total = (K_red + 63) / 64, T_total = N_out / 32;
    PanelTail t;
    // (the result's columns reach their channels from the product itself, or in a pass of their own when there are many)
    const bool scatter = trans && xsrc && (plan.split_k > 1 || panel_scatters(M, K));
    t.bias = bias, t.y = scatter ? xs : y, t.partial = partial, t.out_map = trans && !scatter ? xsrc : nullptr;
    t.G = K / group_size;
    t.q_bytes = (uint32_t)((unsigned long long)T_total * S_total * 256 * bits);
    t.s_bytes = trans ? (uint32_t)t.G * (uint32_t)S_total * 256u : (uint32_t)t.G * (uint32_t)N * 4u;
    const int main_rbs = plan.split_k > 1 ? panel_main_blocks(plan) : 0, tail0 = 32 * plan.row_tiles * main_rbs;
    t.col_wgs = plan.grid_x, t.main_rbs = main_rbs, t.tail_rbs = plan.m_blocks - main_rbs, t.split_k = plan.split_k, t.tail_steps = plan.k_chunk;
    t.lb_per_group = group_size / 32;
    const uint32_t lbg = (uint32_t)t.lb_per_group, pair = 2u * panel_waves_k(plan.row_tiles), tail_wgs = (uint32_t)(t.col_wgs * t.tail_rbs);
    const unsigned long long wgs = (unsigned long long)t.col_wgs * plan.m_blocks;
    t.column_group_magic = panel_magic(wgs, 4u * t.col_wgs), t.tail_magic = panel_magic((unsigned long long)tail_wgs * t.split_k, tail_wgs);
    t.lb_magic = panel_magic(2ull * S_total + 64, lbg), t.tile_magic = panel_magic(T_total, lbg);
    t.step_groups = pair / lbg, t.step_rem = pair % lbg;
    int rc = GPTQ_HIP_ERR_BAD_ARG;
    auto go = [&](auto bits_c) {
        constexpr int B = decltype(bits_c)::value;
        return trans ? launch_panel_bits<B, true>((const _Float16 *)x, (const char *)qtile, sz, M, K_red, N_out, S_total, T_total, t, plan, stream)
                     : launch_panel_bits<B, false>((const _Float16 *)x, (const char *)qtile, sz, M, K_red, N_out, S_total, T_total, t, plan, stream);
    };
    switch (bits) {
        case 2: rc = go(std::integral_constant<int, 2>{}); break;
        case 3: rc = go(std::integral_constant<int, 3>{}); break;
        case 4: rc = go(std::integral_constant<int, 4>{}); break;
        case 8: rc = go(std::integral_constant<int, 8>{}); break;
        default: break;
    }
    if (rc != GPTQ_HIP_OK) return rc;
    if (scatter) return launch_panel_scatter(xs, plan.split_k > 1 ? partial : nullptr, xsrc, y, M, K, plan.split_k, tail0, stream);
    if (plan.split_k == 1) return GPTQ_HIP_OK;
    return launch_tiled_reduce(partial, bias, (_Float16 *)y + (size_t)tail0 * N_out, M - tail0, N_out, plan.split_k, nullptr, stream);
}

}  // namespace gptq
