// Page encoder, deterministic raw-slot assignment, device-side append and the
// compressed -> bf16 decoder, for gfx950.
//
// Encoding one call's pages takes two launches on the caller's stream up to 65,536 units (the
// page kernel, then scan_direct_kernel for 2-4 below; fewer where the rowmasks lie scattered or
// unaligned, direct_units()); above, four, or two when the caller gives a scan workspace (2-4 then
// run as one chained scan kernel, scan_chain_kernel):
//   1. enc_pages_kernel    one wavefront per (sequence, page, head): exponent window,
//                          zero flag, codes, sign|mantissa bytes, base bytes, rowmask
//                          (reference kernels.py:216-264, codec.py:31-49);
//   2. scan_count_kernel   per block of 1024 units, its raw rows;
//   3. scan_blocks_kernel  the block totals scanned from the counter, which advances
//                          by the total;
//   4. scan_write_kernel   rowoff = counter + exclusive running count of raw rows over
//                          the call's pages in (sequence, page, head) order (codec.py:50-53
//                          order; the reference GPU encoder used an atomic counter,
//                          kernels.py:262), then the raw rows into their slots, skipping
//                          slots >= cap (kernels.py:265-268), so an overflow is seen from
//                          the counter.
// The append path (cache.py:100-112) is one launch (row writes; at page ends the page encode,
// the slot scan and the raw-row copies) with the token count read from device memory, so a
// decode step can be captured in a HIP graph. Every kernel that touches rows is a template on the
// head dim (64, 128 or 256); the entry points pick the instance.
#include <type_traits>

#include "tile.hpp"
#include "../../include/exactkv.h"

namespace exkv {

__device__ inline uint8_t sm_byte(uint32_t u) { return (uint8_t)(((u >> 8) & 0x80u) | (u & 0x7Fu)); }

// Two 16-bit lanes in one register: the page encoder keeps two channels' exponents per
// register and works on both with packed integer ops (max, min, saturating subtract).
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ inline u16x2 as_u16x2(uint32_t x) { return __builtin_bit_cast(u16x2, x); }
__device__ inline uint32_t as_u32(u16x2 x) { return __builtin_bit_cast(uint32_t, x); }
__device__ inline u16x2 vmax(u16x2 a, u16x2 b) { return __builtin_elementwise_max(a, b); }
__device__ inline u16x2 vmin(u16x2 a, u16x2 b) { return __builtin_elementwise_min(a, b); }
__device__ inline u16x2 vsubs(u16x2 a, u16x2 b) { return __builtin_elementwise_sub_sat(a, b); }   // max(a - b, 0)
// bytes 0 and 2 of x as a 16-bit value
__device__ inline uint16_t bytes02(uint32_t x) { return (uint16_t)__builtin_amdgcn_perm(0u, x, 0x0c0c0200u); }

// Encode one 16-token page of one head of D channels (D = 64, 128, 256). The lanes form
// NG token groups (2; 4 for D = 64) of CL = 64 / NG lanes: lane (grp, m) takes tokens
// TPL*grp .. TPL*grp + TPL - 1 (TPL = 16 / NG) and, in pass p, channels c, c + 1 (word lo)
// and c + D/2, c + D/2 + 1 (word hi) with c = 2 CL p + 2m -- so each code byte (channel j
// low nibble, j + D/2 high nibble) and each pair of sm / code bytes is produced by one
// lane, and every load and store moves two channels (one pass for D <= 128, two for 256).
// Per channel, with e the 8-bit exponent:
//   top = max e over the 16 tokens, floor = max(top - 15, 0), zf = (some e == 0) && floor > 0,
//   nibble = max(e - floor, 0) (e <= top keeps it <= 15; e == 0 gives 0 either way),
//   a row is raw if some channel has e != 0 && e < floor + zf, or if any floor >= 128;
// the same rule as the reference's per-element test (code >= 1 for a non-zero in a
// flagged group, code >= 0 otherwise, floor < 128), in packed 16-bit integer arithmetic.
// The token groups combine their per-channel maxima and minima with one cross-group
// shuffle each (two for four groups). Token p's source row is src + p * s_p, except row
// 15 which comes from `last` when given; rows must be 4-byte aligned (even element
// offsets: callers check). Destination rows of consecutive tokens are `rs` rows apart
// (rs = H).
template <int D>
__device__ __attribute__((always_inline)) inline uint32_t encode_page(const uint16_t* src, int64_t s_p,
                                                                  const uint16_t* last, int lane,
                                                                  uint8_t* sm0, uint8_t* code0, int64_t rs,
                                                                  uint8_t* basep, int32_t* rmaskp) {
    static_assert(D == 64 || D == 128 || D == 256, "head dim 64, 128 or 256");
    constexpr int NG = D == 64 ? 4 : 2;            // token groups
    constexpr int TPL = kPage / NG;                // tokens per lane
    constexpr int CL = 64 / NG;                    // lanes per group = channel pairs per pass
    constexpr int HALF = D / 2;
    constexpr int NPASS = HALF / (2 * CL);
    const int grp = lane / CL, m = lane % CL;
    const int64_t sm_stride = rs * D, code_stride = rs * HALF;
    uint32_t esc = 0;                              // bit i: token TPL*grp + i escapes
    bool big = false;
#pragma unroll
    for (int pass = 0; pass < NPASS; ++pass) {
        const int c = 2 * CL * pass + 2 * m;
        // per-lane row-0 addresses of the lane's group; token i of the group is i strides on
        const uint16_t* srow = src + (int64_t)(TPL * grp) * s_p + c;
        uint8_t* smrow = sm0 + (int64_t)(TPL * grp) * sm_stride + c;
        uint8_t* coderow = code0 + (int64_t)(TPL * grp) * code_stride + c;
        uint32_t lo[TPL], hi[TPL];                 // bf16 pairs: channels (c, c+1), (c+D/2, c+D/2+1)
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            const uint16_t* rp = (i == TPL - 1 && grp == NG - 1 && last != nullptr) ? last + c : srow + i * s_p;
            lo[i] = *reinterpret_cast<const uint32_t*>(rp);
            hi[i] = *reinterpret_cast<const uint32_t*>(rp + HALF);
        }
        u16x2 elo[TPL], ehi[TPL];                  // exponents, one channel per 16-bit lane
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            elo[i] = as_u16x2((lo[i] >> 7) & 0x00FF00FFu);
            ehi[i] = as_u16x2((hi[i] >> 7) & 0x00FF00FFu);
        }
        u16x2 tlo = elo[0], thi = ehi[0], nlo = elo[0], nhi = ehi[0];
#pragma unroll
        for (int i = 1; i < TPL; ++i) {
            tlo = vmax(tlo, elo[i]);
            thi = vmax(thi, ehi[i]);
            nlo = vmin(nlo, elo[i]);
            nhi = vmin(nhi, ehi[i]);
        }
#pragma unroll
        for (int d = CL; d < 64; d <<= 1) {
            tlo = vmax(tlo, as_u16x2((uint32_t)__shfl_xor((int)as_u32(tlo), d)));
            thi = vmax(thi, as_u16x2((uint32_t)__shfl_xor((int)as_u32(thi), d)));
            nlo = vmin(nlo, as_u16x2((uint32_t)__shfl_xor((int)as_u32(nlo), d)));
            nhi = vmin(nhi, as_u16x2((uint32_t)__shfl_xor((int)as_u32(nhi), d)));
        }
        const u16x2 c15 = {15, 15}, one = {1, 1};
        const u16x2 flo = vsubs(tlo, c15), fhi = vsubs(thi, c15);                 // floors
        const u16x2 zlo = vmin(vsubs(one, nlo), vmin(flo, one));                  // zero flags (0 / 1)
        const u16x2 zhi = vmin(vsubs(one, nhi), vmin(fhi, one));
        const u16x2 glo = flo + zlo, ghi = fhi + zhi;                             // non-zero e below: raw
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
            const uint32_t dlo = as_u32(vmin(vsubs(glo, elo[i]), elo[i]));
            const uint32_t dhi = as_u32(vmin(vsubs(ghi, ehi[i]), ehi[i]));
            esc |= (uint32_t)((dlo | dhi) != 0u) << i;
            // code bytes c (nibble of c | nibble of c+D/2 << 4) and c+1 (c+1 | c+1+D/2 << 4)
            const uint32_t cw = as_u32(vsubs(elo[i], flo)) | (as_u32(vsubs(ehi[i], fhi)) << 4);
            // sm bytes: sign over bit 7 of each bf16's mantissa byte
            const uint32_t slo = (lo[i] & 0x007F007Fu) | ((lo[i] >> 8) & 0x00800080u);
            const uint32_t shi = (hi[i] & 0x007F007Fu) | ((hi[i] >> 8) & 0x00800080u);
            uint8_t* sp = smrow + i * sm_stride;
            *reinterpret_cast<uint16_t*>(sp) = bytes02(slo);
            *reinterpret_cast<uint16_t*>(sp + HALF) = bytes02(shi);
            *reinterpret_cast<uint16_t*>(coderow + i * code_stride) = bytes02(cw);
        }
        if (grp == 0) {
            const u16x2 c128 = {128, 128}, c255 = {255, 255};
            const uint32_t blo = as_u32(vmin(flo + zlo * c128, c255)), bhi = as_u32(vmin(fhi + zhi * c128, c255));
            *reinterpret_cast<uint16_t*>(basep + c) = bytes02(blo);
            *reinterpret_cast<uint16_t*>(basep + HALF + c) = bytes02(bhi);
        }
        big = big || ((as_u32(flo) | as_u32(fhi)) & 0xFF80FF80u) != 0u;
    }
    // rowmask: ballot bits [CL*grp, CL*grp + CL) are token TPL*grp + i; a floor of 128 or
    // more in any channel makes every row raw
    uint32_t rm = __ballot(big) != 0 ? 0xFFFFu : 0u;
    constexpr uint64_t kGroup = CL == 64 ? ~0ull : (1ull << CL) - 1ull;
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
        const uint64_t bal = __ballot((esc >> i) & 1u);
#pragma unroll
        for (int gi = 0; gi < NG; ++gi)
            if (((bal >> (CL * gi)) & kGroup) != 0u) rm |= 1u << (TPL * gi + i);
    }
    if (lane == 0 && rmaskp != nullptr) *rmaskp = (int32_t)rm;
    return rm;
}

struct EncArgs {
    const uint16_t* src;
    int64_t s_b, s_pg, s_p, s_h;      // source strides in elements
    uint8_t* sm;
    uint8_t* code;
    uint8_t* base;
    int32_t* rowmask;
    int32_t* rowoff;
    uint16_t* raw;
    int32_t* cnt;
    int32_t* before;
    int64_t cap;
    int b0, pg0, nb, npg, H, TS;
    // Paged destination: page pg of source sequence bi goes to page dst_pages[bi *
    // dst_stride + pg] of the arrays read as B * TS / 16 pages (entries clamped to them);
    // nullptr: page pg0 + pg of sequence b0 + bi.
    const int32_t* dst_pages = nullptr;
    int64_t dst_stride = 0;
    int64_t all_pages = 0;
    int D = kD;                       // head dim: 64, 128 or 256
};

__device__ inline void unit_coords(const EncArgs& a, int64_t u, int& bi, int& pg, int& hk) {
    hk = (int)(u % a.H);
    const int64_t q = u / a.H;
    pg = (int)(q % a.npg);
    bi = (int)(q / a.npg);
}

// Page index of unit (bi, pg) in the arrays read as a list of pages.
__device__ inline int64_t unit_pidx(const EncArgs& a, int bi, int pg) {
    if (a.dst_pages == nullptr) return (int64_t)(a.b0 + bi) * (a.TS / kPage) + (a.pg0 + pg);
    const int32_t e = a.dst_pages[bi * a.dst_stride + pg];
    return (int64_t)min((uint64_t)(uint32_t)e, (uint64_t)(a.all_pages - 1));
}
__device__ inline int64_t unit_page(const EncArgs& a, int bi, int pg, int hk) {
    return unit_pidx(a, bi, pg) * a.H + hk;
}

// One wavefront per unit (sequence, page, head); the unit's coordinates and addresses are
// wavefront-uniform (scalar arithmetic, 32-bit: unit counts are below 2^31).
template <int D>
__global__ void __launch_bounds__(256) enc_pages_kernel(EncArgs a, int nunits) {
    const int lane = threadIdx.x & 63;
    const int u = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (u >= nunits) return;
    const uint32_t q = (uint32_t)u / (uint32_t)a.H, bi = q / (uint32_t)a.npg;
    const int hk = u - (int)(q * (uint32_t)a.H), pg = (int)(q - bi * (uint32_t)a.npg);
    const uint16_t* src = a.src + (int64_t)bi * a.s_b + (int64_t)pg * a.s_pg + (int64_t)hk * a.s_h;
    const int64_t pidx = unit_pidx(a, (int)bi, pg);
    const int64_t row0 = pidx * kPage * a.H + hk, page = pidx * a.H + hk;
    // the raw-row counter as the call finds it, where scan_direct_kernel's blocks read it
    if (u == 0 && lane == 0) a.rowoff[page] = *a.cnt;
    encode_page<D>(src, a.s_p, nullptr, lane, a.sm + row0 * D, a.code + row0 * (D / 2), a.H, a.base + page * D,
                   a.rowmask + page);
}

// The slot scan after a page encode, one unit per thread and 1024 units per block, every
// access coalesced:
//   scan_count_kernel   block g: its units' raw rows -> the rowoff slot of its first unit;
//   scan_blocks_kernel  one workgroup: exclusive scan of the block totals from the
//                       counter -> the same slots; the counter advances by the total;
//   scan_write_kernel   block g: rowoff = its slot's offset + the block's exclusive scan,
//                       then each wavefront copies the raw rows of its escaped units.
// The block totals need no workspace: the slot of a block's first unit is read by that
// block alone, and its final value (the block's offset + 0) is the one read.
constexpr int kScanUnits = 1024;

// Coordinates and page (in the arrays read as pages x heads) of unit u, with the layout
// fixed at compile time (unit counts are below 2^31: the entry points check).
template <bool PAGED>
__device__ inline int64_t unit_page32(const EncArgs& a, int u, int& bi, int& pg, int& hk) {
    const int q = u / a.H;
    hk = u - q * a.H;
    bi = q / a.npg;
    pg = q - bi * a.npg;
    if (PAGED) {
        const int32_t e = a.dst_pages[(int64_t)bi * a.dst_stride + pg];
        return (int64_t)min((uint64_t)(uint32_t)e, (uint64_t)(a.all_pages - 1)) * a.H + hk;
    }
    return ((int64_t)(a.b0 + bi) * (a.TS / kPage) + (a.pg0 + pg)) * a.H + hk;
}

__device__ inline int64_t first_page_of(const EncArgs& a, int64_t g) {
    int bi, pg, hk;
    unit_coords(a, g * kScanUnits, bi, pg, hk);
    return unit_page(a, bi, pg, hk);
}

template <bool PAGED>
__global__ void __launch_bounds__(1024) scan_count_kernel(EncArgs a, int nunits) {
    const int u = blockIdx.x * kScanUnits + threadIdx.x;
    int bi, pg, hk;
    uint32_t m = 0;
    if (u < nunits) m = (uint32_t)a.rowmask[unit_page32<PAGED>(a, u, bi, pg, hk)];
    int total;
    block_excl_scan(popc32(m), total);
    if (threadIdx.x == 0) a.rowoff[first_page_of(a, blockIdx.x)] = total;
}

__global__ void __launch_bounds__(1024) scan_blocks_kernel(EncArgs a, int64_t nblocks) {
    const int64_t per = (nblocks + 1023) / 1024;
    const int64_t g0 = min((int64_t)threadIdx.x * per, nblocks), g1 = min(g0 + per, nblocks);
    const int cnt0 = *a.cnt;
    int local = 0;
    for (int64_t g = g0; g < g1; ++g) local += a.rowoff[first_page_of(a, g)];
    int total;
    int run = cnt0 + block_excl_scan(local, total);
    for (int64_t g = g0; g < g1; ++g) {
        const int64_t p = first_page_of(a, g);
        const int t = a.rowoff[p];
        a.rowoff[p] = run;
        run += t;
    }
    if (threadIdx.x == 0) {
        if (a.before) *a.before = cnt0;
        *a.cnt = cnt0 + total;
    }
}

// The raw rows (D channels) of the escaped units among a wavefront's 64 (lane = unit: mask
// m, first slot off, source row 0 at src). VEC16 (source rows 16-byte aligned): four units
// at a time, a 16-lane group per unit, each lane moving D/16 channels (8 or 16 bytes) of
// every row of its unit per pass (two passes for D = 256) with all the unit's loads of a
// pass in flight; else one unit at a time, 4 bytes of each row per lane per pass. Slots at
// or past cap are skipped (the host grows the pool and encodes again).
template <bool VEC16, int D>
__device__ inline void copy_escaped_rows(const EncArgs& a, uint32_t m, int32_t off, const uint16_t* src,
                                         int lane) {
    uint64_t todo = __ballot(m != 0);
    if (VEC16) {
        constexpr int EPL = D == 64 ? 4 : 8;           // channels per lane per pass
        constexpr int NPASS = D / (16 * EPL);
        const int g = lane >> 4, j = lane & 15;
        while (todo != 0) {
            int pick = -1;                             // group g takes the g-th unit left
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (todo != 0) {
                    if (i == g) pick = __builtin_ctzll(todo);
                    todo &= todo - 1;
                }
            const int from = pick < 0 ? 0 : pick;
            // every lane joins the shuffles (a shuffle from a lane outside the executing
            // ones reads 0): the unit's mask, first slot and source row
            const uint32_t mv = (uint32_t)__shfl((int)m, from);
            const uint32_t mp = pick < 0 ? 0u : mv;
            const int32_t op = __shfl(off, from);
            const uint64_t sp = ((uint64_t)(uint32_t)__shfl((int)(uint32_t)(uintptr_t)src, from)) |
                                ((uint64_t)(uint32_t)__shfl((int)(uint32_t)((uintptr_t)src >> 32), from) << 32);
            const int nr = popc32(mp);
#pragma unroll
            for (int pass = 0; pass < NPASS; ++pass) {
                const int c0 = 16 * EPL * pass + EPL * j;
                const uint16_t* s = reinterpret_cast<const uint16_t*>(sp) + c0;
                uint32_t t = mp;
                uint32_t r[kPage][EPL / 2];
#pragma unroll
                for (int k = 0; k < kPage; ++k) {      // the k-th escaped row of the unit
                    const int p = t != 0u ? __builtin_ctz(t) : 0;
                    t &= t - 1u;
                    if (k < nr) {
                        ld_words<EPL / 2>(s + p * a.s_p, r[k]);
                    } else {
#pragma unroll
                        for (int w = 0; w < EPL / 2; ++w) r[k][w] = 0u;
                    }
                }
#pragma unroll
                for (int k = 0; k < kPage; ++k)
                    if (k < nr && (int64_t)op + k < a.cap) st_words<EPL / 2>(a.raw + ((int64_t)op + k) * D + c0, r[k]);
            }
        }
    } else {
        constexpr int NPASS = D > 128 ? D / 128 : 1;
        while (todo != 0) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t mp = (uint32_t)__builtin_amdgcn_readlane((int)m, l);
            const int32_t op = __builtin_amdgcn_readlane(off, l);
            const uint64_t sp = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uintptr_t)src, l) |
                                ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uintptr_t)src >> 32), l) << 32);
            const int nr = popc32(mp);
#pragma unroll
            for (int pass = 0; pass < NPASS; ++pass) {
                const int c0 = 128 * pass + 2 * lane;
                if (c0 >= D) continue;                 // D = 64: half the lanes
                const uint16_t* s = reinterpret_cast<const uint16_t*>(sp) + c0;
                uint32_t t = mp;
                uint32_t r[kPage];
#pragma unroll
                for (int k = 0; k < kPage; ++k) {
                    const int p = t != 0u ? __builtin_ctz(t) : 0;
                    t &= t - 1u;
                    r[k] = k < nr ? *reinterpret_cast<const uint32_t*>(s + p * a.s_p) : 0u;
                }
#pragma unroll
                for (int k = 0; k < kPage; ++k)
                    if (k < nr && (int64_t)op + k < a.cap)
                        *reinterpret_cast<uint32_t*>(a.raw + ((int64_t)op + k) * D + c0) = r[k];
            }
        }
    }
}

template <bool PAGED, bool VEC16, int D>
__global__ void __launch_bounds__(1024) scan_write_kernel(EncArgs a, int nunits) {
    __shared__ int s_base;
    if (threadIdx.x == 0) s_base = a.rowoff[first_page_of(a, blockIdx.x)];
    const int u = blockIdx.x * kScanUnits + threadIdx.x;
    int bi = 0, pg = 0, hk = 0;
    int64_t page = 0;
    uint32_t m = 0;
    if (u < nunits) {
        page = unit_page32<PAGED>(a, u, bi, pg, hk);
        m = (uint32_t)a.rowmask[page];
    }
    int total;
    const int off = block_excl_scan(popc32(m), total) + s_base;   // synchronises: s_base is read
    if (u < nunits) a.rowoff[page] = off;
    copy_escaped_rows<VEC16, D>(a, m, off, a.src + bi * a.s_b + pg * a.s_pg + hk * a.s_h, threadIdx.x & 63);
}

// Whether every source row starts at a multiple of 16 bytes.
static bool rows_of_16_bytes(const EncArgs& a) {
    return (uintptr_t)a.src % 16 == 0 && a.s_b % 8 == 0 && a.s_pg % 8 == 0 && a.s_p % 8 == 0 && a.s_h % 8 == 0;
}

template <int D>
static void launch_scan(const EncArgs& a, int64_t n, hipStream_t stream) {
    const unsigned nb = (unsigned)((n + kScanUnits - 1) / kScanUnits);
    const bool paged = a.dst_pages != nullptr, vec16 = rows_of_16_bytes(a);
    if (paged)
        hipLaunchKernelGGL(scan_count_kernel<true>, dim3(nb), dim3(1024), 0, stream, a, (int)n);
    else
        hipLaunchKernelGGL(scan_count_kernel<false>, dim3(nb), dim3(1024), 0, stream, a, (int)n);
    hipLaunchKernelGGL(scan_blocks_kernel, dim3(1), dim3(1024), 0, stream, a, (int64_t)nb);
    auto k = paged ? (vec16 ? scan_write_kernel<true, true, D> : scan_write_kernel<true, false, D>)
                   : (vec16 ? scan_write_kernel<false, true, D> : scan_write_kernel<false, false, D>);
    hipLaunchKernelGGL(k, dim3(nb), dim3(1024), 0, stream, a, (int)n);
}

// ---- two-launch encode: the page kernel, then one scan kernel whose blocks chain
//
// scan_chain_kernel: block = kScanUnits units, as scan_write_kernel, but the blocks take
// their places in ticket order (an atomic counter, so that every block's predecessors have
// started) and chain their raw-row totals with a decoupled look-back (Merrill & Garland,
// "Single-pass Parallel Prefix Scan with Decoupled Look-back", NVIDIA technical report
// NVR-2016-002): a block publishes its total, walks back over its predecessors' published
// words until one that already includes everything before it, and publishes its inclusive
// total. Block 0 starts from the pool counter; the last block writes the counter back.
// rowoff, raw slots and counter come out exactly as from the three-launch scan.
//
// Workspace (the caller's; all zero when first used, then only this kernel writes it):
// ws[0] the ticket counter, ws[1] a call generation, ws[2 + t] block t's word: the call's
// tag (bits 63-32: the generation's low 31 bits with bit 63 set, so that neither words
// left by earlier calls nor never-written zero words are taken for this call's), inclusive
// flag (bit 31), count (bits 30-0). The last ticket holder resets the counter and advances
// the generation, so consecutive calls on one stream share a workspace; calls that
// overlap on one workspace race.
constexpr uint64_t kInclusive = 1ull << 31;
constexpr int kLookbackSpin = 1 << 22;              // bound of the look-back's waits (never reached; reported)

__device__ inline uint64_t ws_ld(const uint64_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void ws_st(uint64_t* p, uint64_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline uint32_t chain_tag(uint32_t gen) { return (gen & 0x7FFFFFFFu) | 0x80000000u; }

// Exclusive prefix of block `t0 + 1` (t0 >= 0): one wavefront reads 64 predecessors' words
// at a time (lane i: block t - i), nearest first; every word up to the nearest inclusive one
// must carry this call's tag (else the window is read again), and their counts are summed.
__device__ inline int64_t chain_lookback(const uint64_t* ws, uint32_t tag, int t0, int lane) {
    int64_t excl = 0;
    int t = t0;
    for (int s = 0; s < kLookbackSpin; ++s) {
        const int tt = t - lane;
        const uint64_t st = tt >= 0 ? ws_ld(ws + 2 + tt) : (((uint64_t)tag << 32) | kInclusive);
        const bool valid = (uint32_t)(st >> 32) == tag;
        const uint64_t incl = __ballot(valid && (st & kInclusive) != 0);
        const int stop = incl != 0 ? __builtin_ctzll(incl) : 63;
        const uint64_t need = stop == 63 ? ~0ull : (2ull << stop) - 1ull;
        if ((~__ballot(valid) & need) != 0) {          // a predecessor has not published yet
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        // block totals (<= 16 * kScanUnits each) summed in 32 bits, the inclusive word apart
        int v = lane < stop || (incl == 0 && lane == stop) ? (int)(st & 0x7FFFFFFFull) : 0;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) v += __shfl_xor(v, d);
        excl += v;
        if (incl != 0)
            return excl + (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(st & 0x7FFFFFFFull), stop);
        t -= 64;
    }
    if (lane == 0) report_error(kErrLookback);          // gave up: the prefix is partial
    return excl;
}

template <bool PAGED, bool VEC16, int D>
__global__ void __launch_bounds__(1024) scan_chain_kernel(EncArgs a, int nunits, int nblocks, uint64_t* ws) {
    __shared__ int s_tile, s_excl;
    __shared__ uint32_t s_gen;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) {
        const uint32_t gen = (uint32_t)ws_ld(ws + 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the generation is read before the ticket is taken
        const uint32_t t = __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(ws), 1u, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
        if (t == (uint32_t)nblocks - 1u) {             // every ticket of this call is out
            ws_st(ws, 0ull);
            ws_st(ws + 1, (uint64_t)(gen + 1u));
        }
        s_tile = (int)t;
        s_gen = gen;
    }
    __syncthreads();
    const int tile = s_tile;
    const uint32_t tag = chain_tag(s_gen);
    if ((uint32_t)tile >= (uint32_t)nblocks) {         // a workspace left inconsistent (misuse): write nothing
        if (threadIdx.x == 0) report_error(kErrScanWs);
        return;
    }
    const int u = tile * kScanUnits + threadIdx.x;
    int bi = 0, pg = 0, hk = 0;
    int64_t page = 0;
    uint32_t m = 0;
    if (u < nunits) {
        page = unit_page32<PAGED>(a, u, bi, pg, hk);
        m = (uint32_t)a.rowmask[page];
    }
    int total;
    const int pre = block_excl_scan(popc32(m), total);   // synchronises
    if (threadIdx.x < 64) {
        int64_t excl;
        if (tile == 0) {
            excl = *a.cnt;
            if (lane == 0 && a.before != nullptr) *a.before = (int32_t)excl;
        } else {
            if (lane == 0) ws_st(ws + 2 + tile, ((uint64_t)tag << 32) | (uint32_t)total);
            excl = chain_lookback(ws, tag, tile - 1, lane);
        }
        if (lane == 0) {
            ws_st(ws + 2 + tile, ((uint64_t)tag << 32) | kInclusive | (uint64_t)(uint32_t)(excl + total));
            if (tile == nblocks - 1) *a.cnt = (int32_t)(excl + total);
            s_excl = (int)excl;
        }
    }
    __syncthreads();
    const int off = s_excl + pre;
    if (u < nunits) a.rowoff[page] = off;
    copy_escaped_rows<VEC16, D>(a, m, off, a.src + bi * a.s_b + pg * a.s_pg + hk * a.s_h, lane);
}

// ---- two-launch encode of up to kDirectUnits units: no block waits for another
//
// scan_direct_kernel: block of `ub` units; it counts the raw rows of every unit before its own
// by reading their rowmasks again (4 bytes a unit, from the L2s the page kernel left them in),
// so all blocks start at once and need neither tickets nor a workspace. The counter's value
// before the call comes from the rowoff slot of the call's first unit, where the page kernel
// put it and whose final value it is; the last block, which has counted every unit, writes the
// counter back. The blocks are small (64 units up to 16,384, so that a 4,096-token slot of 8
// heads runs 32 of them instead of the chain's 2 of 1,024) and their 16 wavefronts take 4 to
// 16 units each, which is what the raw-row copies need: their loads are a dependent round
// trip after the masks. The masks read grow with the square of the units (33 MB at 65,536, in
// 256 blocks), hence the limit; where they can't be read four at a time (a block table, or
// masks that are not 16-byte aligned) a mask costs two divisions, and with a table a load before
// its own, so the line lies where the chain gets ahead: encodes direct / chained at head dim 128
// through a table, 8,192 units 20.0 / 21.2 us, 10,240 23.0 / 23.4, 16,384 32.8 / 30.6, 65,536
// 132.4 / 102.7; unaligned, 10,240 21.5 / 22.8, 12,288 24.5 / 24.9, 16,384 30.0 / 29.3, 65,536
// 118.0 / 98.0 (head dim 64 crosses at 8,192 and 12,288). A prefill's end rides in the direct
// scan's launch and needs one of its own beside the chain: a paged slot of 10,000 units 43.0 /
// 46.2, 16,376 53.7 / 53.9, 30,000 75.2 / 64.7.
constexpr int kDirectUnits = 65536, kDirectUnitsUnaligned = 12288, kDirectUnitsPaged = 8192;
constexpr int kDirectUnitsPrefill = 16384;             // with a prefill's end, of masks read one by one

// Whether the masks of the call's units lie in rows whose parts of four words are 16-byte aligned.
__host__ __device__ inline bool masks_by_four(const EncArgs& a) {
    if (a.dst_pages != nullptr) return false;
    const int64_t L = (int64_t)a.npg * a.H, S = (int64_t)(a.TS / kPage) * a.H;   // words a sequence, and to the next
    return (uintptr_t)(a.rowmask + a.b0 * S + (int64_t)a.pg0 * a.H) % 16 == 0 && (a.nb == 1 || (L % 4 == 0 && S % 4 == 0));
}

static int direct_units(const EncArgs& a, bool prefill) {
    if (masks_by_four(a)) return kDirectUnits;
    return prefill ? kDirectUnitsPrefill : a.dst_pages != nullptr ? kDirectUnitsPaged : kDirectUnitsUnaligned;
}

static int direct_block_units(int64_t n) { return n <= 16384 ? 64 : n <= 32768 ? 128 : 256; }

// Raw rows of units [0, u0), this thread's share (1,024 threads, all of them calling). u0 is a
// multiple of 64.
template <bool PAGED>
__device__ inline int raw_rows_before(const EncArgs& a, int u0) {
    int sum = 0;
    if (!PAGED) {
        const int L = a.npg * a.H;                     // a sequence's masks: L words in a row, every S words
        const int64_t S = (int64_t)(a.TS / kPage) * a.H;
        const int32_t* p0 = a.rowmask + (int64_t)a.b0 * S + (int64_t)a.pg0 * a.H;
        const bool one = a.nb == 1;
        if (masks_by_four(a)) {                        // uniform
            for (int v0 = 4 * (int)threadIdx.x; v0 < u0; v0 += 4 * 4096) {
                uint4 m[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int v = v0 + 4096 * k;
                    m[k] = make_uint4(0u, 0u, 0u, 0u);
                    if (v < u0) {
                        const int bi = one ? 0 : v / L;
                        m[k] = *reinterpret_cast<const uint4*>(p0 + bi * S + (v - bi * L));
                    }
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) sum += popc32(m[k].x) + popc32(m[k].y) + popc32(m[k].z) + popc32(m[k].w);
            }
            return sum;
        }
    }
    for (int v0 = threadIdx.x; v0 < u0; v0 += 4 * 1024) {
        uint32_t m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int v = v0 + 1024 * k;
            int bi, pg, hk;
            m[k] = v < u0 ? (uint32_t)a.rowmask[unit_page32<PAGED>(a, v, bi, pg, hk)] : 0u;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) sum += popc32(m[k]);
    }
    return sum;
}

// What a prefill does besides encoding its full pages: the rows of its last, partly filled page
// go to the slot's open-page rows, that page is opened, and the device token count is set. One
// more block of the scan's launch does it beside the scan, in its shadow (30 KB of rows at 8
// heads of 128), instead of a fill, a strided copy and an open-page launch, the last two after
// the host's wait for the raw-row counter: a layer's K and V of a 4,091-token prompt
// 122 -> 61 us, of which the GPU works 2 x 9.
struct PrefillEnd {
    const uint16_t* tail = nullptr;   // token 0 of the open page, head 0 (rows s_t apart, heads s_h)
    int64_t s_t = 0, s_h = 0;
    int rows = 0;                     // its tokens: T % 16
    int64_t tail0 = 0;                // raw row of its token 0, head 0 (heads 16 rows apart)
    int32_t* state = nullptr;         // contiguous: state[0] = T
    int T = 0;
    int B = 0;                        // contiguous: page T / 16 of every sequence is opened
    int open_pages = 0;               // pages per sequence: none is opened at or past it
    const int32_t* table = nullptr;   // paged: the slot's block-table row; its page T / 16 is opened
    int64_t pool_pages = 0;
    int32_t* host = nullptr;          // mapped host memory: the counter to host[1], then tag to host[0]
    int32_t tag = 0;
    int32_t* arrivals = nullptr;      // with host: the scan's blocks count in here (zero between calls)
};

// A word to mapped host memory, past the caches: complete at this wave's next vmcnt(0).
__device__ inline void to_host(int32_t* p, int32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The open page's rows, e.rows x H, in pieces of E channels, by 1,024 threads with up to N
// pieces each in flight. A thread's pieces are 1,024 / (D / E) rows apart: it steps from one to the
// next by additions, since a division for each piece, one piece at a time, was most of the
// prefill where the pieces are many (a call with 15 rows x 128 heads x 256, 4-byte aligned,
// 159 -> 77 us; x 32 x 128 40 -> 32).
template <int D, int E>
__device__ inline void copy_open_rows(const PrefillEnd& e, int H, uint16_t* dst) {
    constexpr int CH = D / E, N = E == 8 ? 4 : 16, W = E == 1 ? 1 : E / 2;
    typedef typename std::conditional<E == 1, uint16_t, uint32_t>::type word;
    const int c = (int)threadIdx.x % CH * E, u = (int)threadIdx.x / CH;
    int r = u / H, h = u % H;
    const int dr = 1024 / CH / H, dh = 1024 / CH % H;      // from a piece to the thread's next
    const int64_t ds = dr * e.s_t + dh * e.s_h, dd = ((int64_t)dh * kPage + dr) * D;
    const int64_t ws = e.s_t - H * e.s_h, wd = (1 - (int64_t)H * kPage) * D;   // and over the last head
    const uint16_t* src = e.tail + r * e.s_t + h * e.s_h + c;
    dst += ((int64_t)h * kPage + r) * D + c;
    while (r < e.rows) {
        word v[N][W];
        uint16_t* at[N];
#pragma unroll
        for (int k = 0; k < N; ++k) {
            at[k] = r < e.rows ? dst : nullptr;
            if (r < e.rows) {
                if constexpr (E == 1) v[k][0] = src[0]; else ld_words<W>(src, v[k]);
            }
            const bool over = h + dh >= H;
            r += dr + over;
            h += over ? dh - H : dh;
            src += ds + (over ? ws : 0);
            dst += dd + (over ? wd : 0);
        }
#pragma unroll
        for (int k = 0; k < N; ++k)
            if (at[k] != nullptr) {
                if constexpr (E == 1) at[k][0] = v[k][0]; else st_words<W>(at[k], v[k]);
            }
    }
}

// One block of 1,024 threads.
template <int D>
__device__ inline void prefill_end(const EncArgs& a, const PrefillEnd& e) {
    const int pg = e.T / kPage, H = a.H;
    if (pg < e.open_pages) {
        if (e.table != nullptr) {
            const int64_t pidx = min((uint64_t)(uint32_t)e.table[pg], (uint64_t)(e.pool_pages - 1));
            for (int h = threadIdx.x; h < H; h += 1024) {
                a.rowmask[pidx * H + h] = 0xFFFF;
                a.rowoff[pidx * H + h] = (int32_t)(e.tail0 + (int64_t)h * kPage);
            }
        } else {
            for (int u = threadIdx.x; u < e.B * H; u += 1024) {
                const int64_t page = ((int64_t)(u / H) * e.open_pages + pg) * H + u % H;
                a.rowmask[page] = 0xFFFF;
                a.rowoff[page] = (int32_t)(a.cap + (int64_t)u * kPage);
            }
        }
    }
    if (e.state != nullptr && threadIdx.x == 0) e.state[0] = e.T;
    uint16_t* dst = a.raw + e.tail0 * D;
    if ((uintptr_t)e.tail % 16 == 0 && e.s_t % 8 == 0 && e.s_h % 8 == 0)      // uniform
        copy_open_rows<D, 8>(e, H, dst);
    else if ((uintptr_t)e.tail % 4 == 0 && e.s_t % 2 == 0 && e.s_h % 2 == 0)
        copy_open_rows<D, 2>(e, H, dst);
    else
        copy_open_rows<D, 1>(e, H, dst);
}

// A prefill's end by itself: a prompt of less than a page, or one too long for the direct scan.
template <int D>
__global__ void __launch_bounds__(1024) prefill_end_kernel(EncArgs a, PrefillEnd e) {
    prefill_end<D>(a, e);
    if (e.host == nullptr) return;                     // uniform
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        to_host(e.host + 1, *a.cnt);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        to_host(e.host, e.tag);
    }
}

// Count this block in on *arrivals (zero between calls): true for the last of the grid's. Every
// thread calls it; a wave's loads and stores are complete first (stores: it waits for them).
__device__ inline bool last_block(int32_t* arrivals, bool stores) {
    __shared__ int s_last;
    if (stores) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const int old = __hip_atomic_fetch_add(arrivals, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = old == (int)gridDim.x - 1;
    }
    __syncthreads();
    return s_last != 0;
}

// The last block to arrive, after the block with the counter's value has stored it and every
// block has read its rows, tells the host, which waits for that: a launch of its own for it took
// 1 us more of a prefill at every size (one cache, with its counter's fill: 2,045 units 28.4 ->
// 27.2 us, 8,190 35.7 -> 34.7, 32,760 in 257 blocks 63.2 -> 62.5).
__device__ inline void tell_host(const PrefillEnd& e) {
    if (e.host == nullptr) return;                     // uniform
    if (last_block(e.arrivals, true) && threadIdx.x == 0) {
        __hip_atomic_store(e.arrivals, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        to_host(e.host, e.tag);
    }
}

// nscan blocks of ub units; END: one more, which does a prefill's end beside them.
template <bool PAGED, bool VEC16, bool END, int D>
__global__ void __launch_bounds__(1024) scan_direct_kernel(EncArgs a, int nunits, int ub, int nscan, PrefillEnd e) {
    if (END && (int)blockIdx.x == nscan) {
        prefill_end<D>(a, e);
        tell_host(e);
        return;
    }
    __shared__ int s_before[16], s_own[16];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, per = ub >> 4;   // units per wavefront
    const int u0 = (int)blockIdx.x * ub, u = u0 + w * per + lane;
    int bi = 0, pg = 0, hk = 0;
    const int cnt0 = a.rowoff[unit_page32<PAGED>(a, 0, bi, pg, hk)];
    int64_t page = 0;
    uint32_t m = 0;
    const bool mine = lane < per && u < nunits;
    if (mine) {
        page = unit_page32<PAGED>(a, u, bi, pg, hk);
        m = (uint32_t)a.rowmask[page];
    }
    const int before = wave_incl_scan(raw_rows_before<PAGED>(a, u0));
    const int own = wave_incl_scan(popc32(m));
    if (lane == 63) {
        s_before[w] = before;
        s_own[w] = own;
    }
    __syncthreads();
    int pre = cnt0, total = 0;                         // rows before this wavefront's units; the block's
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        pre += s_before[i] + (i < w ? s_own[i] : 0);
        total += s_before[i] + s_own[i];
    }
    const int off = pre + own - popc32(m);
    if (mine) a.rowoff[page] = off;
    if (threadIdx.x == 0) {
        if (blockIdx.x == 0 && a.before != nullptr) *a.before = cnt0;
        if ((int)blockIdx.x == nscan - 1) {
            *a.cnt = cnt0 + total;
            if (END && e.host != nullptr) to_host(e.host + 1, cnt0 + total);
        }
    }
    if (a.cap > 0) copy_escaped_rows<VEC16, D>(a, m, off, a.src + bi * a.s_b + pg * a.s_pg + hk * a.s_h, lane);
    if (END) tell_host(e);
}

template <int D, bool END>
static void launch_direct(const EncArgs& a, int64_t n, bool paged, bool vec16, const PrefillEnd& e, hipStream_t stream) {
    const int ub = direct_block_units(n), nscan = (int)((n + ub - 1) / ub);
    auto k = paged ? (vec16 ? scan_direct_kernel<true, true, END, D> : scan_direct_kernel<true, false, END, D>)
                   : (vec16 ? scan_direct_kernel<false, true, END, D> : scan_direct_kernel<false, false, END, D>);
    hipLaunchKernelGGL(k, dim3((unsigned)(nscan + END)), dim3(1024), 0, stream, a, (int)n, ub, nscan, e);
}

// Encode n units: the page kernel, then the direct scan up to direct_units() units; above, the
// chained scan when the workspace has at least 2 + ceil(n / kScanUnits) words, else the
// three-launch scan. end: a prefill's end too, in the direct scan's launch or in one of its own.
template <int D>
static void launch_encode_d(const EncArgs& a, int64_t n, uint64_t* ws, int64_t ws_words, const PrefillEnd* end,
                            hipStream_t stream) {
    if (n == 0) {
        if (end) hipLaunchKernelGGL(prefill_end_kernel<D>, dim3(1), dim3(1024), 0, stream, a, *end);
        return;
    }
    hipLaunchKernelGGL(enc_pages_kernel<D>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream, a, (int)n);
    const bool paged = a.dst_pages != nullptr, vec16 = rows_of_16_bytes(a);
    if (n <= direct_units(a, end != nullptr)) {
        if (end)
            launch_direct<D, true>(a, n, paged, vec16, *end, stream);
        else
            launch_direct<D, false>(a, n, paged, vec16, PrefillEnd{}, stream);
        return;
    }
    const int64_t nb = (n + kScanUnits - 1) / kScanUnits;
    if (ws == nullptr || ws_words < 2 + nb) {
        launch_scan<D>(a, n, stream);
    } else {
        auto k = paged ? (vec16 ? scan_chain_kernel<true, true, D> : scan_chain_kernel<true, false, D>)
                       : (vec16 ? scan_chain_kernel<false, true, D> : scan_chain_kernel<false, false, D>);
        hipLaunchKernelGGL(k, dim3((unsigned)nb), dim3(kScanUnits), 0, stream, a, (int)n, (int)nb, ws);
    }
    if (end) hipLaunchKernelGGL(prefill_end_kernel<D>, dim3(1), dim3(1024), 0, stream, a, *end);
}

static void launch_encode(const EncArgs& a, int64_t n, uint64_t* ws, int64_t ws_words, const PrefillEnd* end,
                          hipStream_t stream) {
    if (a.D == 64)
        launch_encode_d<64>(a, n, ws, ws_words, end, stream);
    else if (a.D == 256)
        launch_encode_d<256>(a, n, ws, ws_words, end, stream);
    else
        launch_encode_d<128>(a, n, ws, ws_words, end, stream);
}

// The raw rows of pages that are already encoded (rowmask and rowoff in place) into their slots:
// what a call whose pool was too small, or of size 0 to count the rows first, has left to do. A
// wavefront takes kStoreUnits units, so that the copies, each a dependent round trip after the
// masks, spread over the chip; encoding the pages again for it was as long as the first time
// (16 x 4096 tokens x 8 heads: 49 us against 4.7).
constexpr int kStoreUnits = 16;

template <bool VEC16, int D>
__global__ void __launch_bounds__(256) store_raw_kernel(EncArgs a, int nunits) {
    const int lane = threadIdx.x & 63;
    const int u = ((int)blockIdx.x * 4 + (int)(threadIdx.x >> 6)) * kStoreUnits + lane;
    int bi = 0, pg = 0, hk = 0;
    uint32_t m = 0;
    int32_t off = 0;
    if (lane < kStoreUnits && u < nunits) {
        const int64_t page = unit_page32<false>(a, u, bi, pg, hk);
        m = (uint32_t)a.rowmask[page];
        off = a.rowoff[page];
        if (off < 0) m = 0;                            // not this encoder's: outside the pool
    }
    copy_escaped_rows<VEC16, D>(a, m & 0xFFFFu, off, a.src + bi * a.s_b + pg * a.s_pg + hk * a.s_h, lane);
}

// Row of D channels: d[c] = s[c], lanes striding by 64.
template <int D>
__device__ inline void copy_row(uint16_t* d, const uint16_t* s, int lane) {
#pragma unroll
    for (int c = 0; c < D; c += 64) d[c + lane] = s[c + lane];
}

// ---------------------------------------------------------------- device-side append

struct AppendArgs {
    const uint16_t* x;        // [B, H, D] (row strides sx_b, sx_h in elements)
    int64_t sx_b, sx_h;
    uint8_t* sm;
    uint8_t* code;
    uint8_t* base;
    int32_t* rowmask;
    int32_t* rowoff;
    uint16_t* raw;
    int32_t* cnt;
    int32_t* before;
    int32_t* state;           // state[0] = tokens held (T)
    int64_t cap;
    int B, H, TS;
};

// One append in one launch. Each wavefront takes (sequence, head) units u = its index,
// + the grid's wavefronts, ...: it writes the token into the unit's open page (the tail
// area) and, when the token completes page T/16, encodes the page (its rowmask stored
// device-coherently, for the last block) and opens the next one (rowmask all ones, rowoff
// into the tail area). Every block then counts itself in on state[1] (zero between calls)
// once its stores are complete; the last block to arrive -- which therefore follows every
// block's rowmask stores -- assigns the page's raw-row slots by an exclusive scan over the
// units in (sequence, head) order from *cnt (the codec's slot order), copies the raw rows
// (tokens 0-14 from the tail area, written by earlier appends; token 15 from x), sets
// *before and *cnt, and advances state[0]. Replaces three launches (write and encode, slot
// scan, raw-row copy), measured 0.87 ms of a c4 decode step for 64 caches.
//
// ONE: a grid of one block, up to kAppendOne units, where nothing is counted in. An ordinary step
// is then one round trip (the token count and the rows, loaded together) and its stores, and
// is bound by those and the launch. Back-to-back launches, one wavefront per row of 2-byte
// lanes and a count in every step / now: 8 units 3.6 / 2.0 us, 64 4.4 / 2.35, 128 4.8 / 3.2 (8
// blocks), 4,960 5.7 / 4.0. At a page end a block's 16 wavefronts encode its pages in turn (64
// units 10-13 us in four blocks, 15-17 in one, one step in 16), hence the limit.
constexpr int kAppendThreads = 1024;
constexpr int kAppendWaves = kAppendThreads / 64;
// At most this many blocks: every block's arrival is an atomic on one word, and those
// serialise (measured at c4, 64 caches per step: 256 blocks 10.2 us per launch); the
// waves loop over the units instead.
constexpr int kAppendBlocks = 64;
constexpr int kAppendOne = 64;

__device__ inline void st_dev_i32(int32_t* p, int32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline int32_t ld_dev_i32(const int32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One raw row into the pool by one thread: src 4-byte aligned (x rows) or 16 (tail rows).
template <int D>
__device__ inline void copy_row_thread(uint16_t* dst, const uint16_t* src) {
    if (((uintptr_t)src & 15u) == 0) {
        for (int c0 = 0; c0 < 2 * D / 16; c0 += 8) {   // 16-byte pieces, eight in flight
            uint4 v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = reinterpret_cast<const uint4*>(src)[c0 + c];
#pragma unroll
            for (int c = 0; c < 8; ++c)                // registers, not a copy through the stack
                asm volatile("" : "+v"(v[c].x), "+v"(v[c].y), "+v"(v[c].z), "+v"(v[c].w));
#pragma unroll
            for (int c = 0; c < 8; ++c) reinterpret_cast<uint4*>(dst)[c0 + c] = v[c];
        }
    } else {
        for (int c0 = 0; c0 < D / 2; c0 += 16) {       // dwords, sixteen in flight
            uint32_t v[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) v[c] = reinterpret_cast<const uint32_t*>(src)[c0 + c];
#pragma unroll
            for (int c = 0; c < 16; ++c) asm volatile("" : "+v"(v[c]));
#pragma unroll
            for (int c = 0; c < 16; ++c) reinterpret_cast<uint32_t*>(dst)[c0 + c] = v[c];
        }
    }
}

// Raw-row slots and rows of n units whose pages have just been encoded (all kAppendThreads
// threads of one block call it), in unit order from slot cnt0 on: `units` gives the index of a
// unit's page and the source of its row r. Thread t takes
// units [t * per, (t + 1) * per): their rowmasks (device-coherent loads, eight in flight),
// the block's exclusive scan of their raw-row counts (the codec's slot order),
// rowoff. Then the raw rows (rows 0-14 from the unit's tail area, written by earlier
// appends; row 15 from x): with up to LDSU units, spread over the threads one row
// each -- the units' first raw-row ranks go to LDS and the thread holding raw row g finds its
// unit by binary search -- so that a page end costs about one round trip; with more units,
// each thread moves its own units' rows. Rows at or past cap are not written (the counter
// shows the overflow). Returns the number of raw rows.
constexpr int kAppendLdsUnits = 8192;

struct RawPool {
    const int32_t* rowmask;
    int32_t* rowoff;
    uint16_t* raw;
    int64_t cap;
};

template <int D, int LDSU, class Units>
__device__ inline int place_raw_rows(const Units& units, int n, int cnt0, const RawPool& pool) {
    __shared__ int s_rank[LDSU + 1];
    __shared__ uint16_t s_mask[LDSU];
    const int per = (n + kAppendThreads - 1) / kAppendThreads;
    const int u0 = min((int)threadIdx.x * per, n), u1 = min(u0 + per, n);
    const bool table = n <= LDSU;                     // uniform
    int local = 0;
    uint32_t m[8];
    auto masks = [&](int c0) {
#pragma unroll
        for (int k = 0; k < 8; ++k) m[k] = c0 + k < u1 ? (uint32_t)ld_dev_i32(pool.rowmask + units.page(c0 + k)) : 0u;
    };
    for (int c0 = u0; c0 < u1; c0 += 8) {
        masks(c0);
#pragma unroll
        for (int k = 0; k < 8; ++k) local += popc32(m[k]);
    }
    int total;
    int run = block_excl_scan(local, total);
    for (int c0 = u0; c0 < u1; c0 += 8) {
        if (per > 8) masks(c0);                        // else still held
        for (int k = 0; k < 8 && c0 + k < u1; ++k) {
            const int u = c0 + k;
            pool.rowoff[units.page(u)] = cnt0 + run;
            if (table) {
                s_rank[u] = run;
                s_mask[u] = (uint16_t)m[k];
            } else {
                int j = 0;
                for (int r = 0; r < kPage; ++r)
                    if ((m[k] >> r) & 1u) {
                        const int64_t slot = (int64_t)cnt0 + run + j++;
                        if (slot < pool.cap) copy_row_thread<D>(pool.raw + slot * D, units.src_row(u, r));
                    }
            }
            run += popc32(m[k]);
        }
    }
    if (table) {
        if (threadIdx.x == 0) s_rank[n] = total;
        __syncthreads();
        for (int g = threadIdx.x; g < total && (int64_t)cnt0 + g < pool.cap; g += kAppendThreads) {
            int lo = 0, hi = n - 1;                    // the unit u with s_rank[u] <= g < s_rank[u + 1]
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (s_rank[mid] <= g) lo = mid; else hi = mid - 1;
            }
            const uint32_t mk = s_mask[lo];
            int k = g - s_rank[lo], r = 0;             // g is the k-th raw row of unit lo's page
            for (; r < kPage - 1; ++r)
                if (((mk >> r) & 1u) && k-- == 0) break;
            copy_row_thread<D>(pool.raw + ((int64_t)cnt0 + g) * D, units.src_row(lo, r));
        }
    }
    return total;
}

// The token rows of n units into their open pages: 16-byte pieces (4-byte ones where the rows of x
// are not 16-byte aligned), one per thread of the grid, up to four with all their loads in
// flight. units: x(u), tail(u) and token(u), the token's index or -1.
template <int D, int E, class Units>
__device__ inline void write_rows(const Units& units, int n, int tid, int nthreads) {
    constexpr int CH = D / E;                          // pieces of E channels per row
    const int total = n * CH;
    for (int i0 = tid; i0 < total; i0 += 4 * nthreads) {
        uint32_t v[4][E / 2];
        int tok[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = min(i0 + k * nthreads, total - 1), u = i / CH;
            if (k > 0 && i0 + k * nthreads >= total) continue;
            ld_words<E / 2>(units.x(u) + i % CH * E, v[k]);
            tok[k] = units.token(u);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = i0 + k * nthreads, u = i / CH;
            if (i < total && tok[k] >= 0) st_words<E / 2>(units.tail(u) + tok[k] % kPage * D + i % CH * E, v[k]);
        }
    }
}

// Units of a contiguous cache's append at token T (-1: a full cache): every page fills at once
template <int D>
struct AppendUnits {
    const AppendArgs& a;
    int T;
    __device__ int token(int) const { return T; }
    __device__ int64_t page(int u) const {
        return ((int64_t)(u / a.H) * (a.TS / kPage) + T / kPage) * a.H + u % a.H;
    }
    __device__ const uint16_t* x(int u) const { return a.x + (u / a.H) * a.sx_b + (u % a.H) * a.sx_h; }
    __device__ uint16_t* tail(int u) const { return a.raw + (a.cap + (int64_t)u * kPage) * D; }
    __device__ const uint16_t* src_row(int u, int r) const { return r == kPage - 1 ? x(u) : tail(u) + r * D; }
};

template <int D, bool ONE>
__global__ void __launch_bounds__(kAppendThreads) append_kernel(AppendArgs a, bool vec16) {
    const int n = a.B * a.H, lane = threadIdx.x & 63;
    const int u0 = (int)blockIdx.x * kAppendWaves + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = (int)gridDim.x * kAppendWaves;
    const int T = a.state[0];
    const AppendUnits<D> units{a, T < a.TS ? T : -1};
    const int tid = (int)blockIdx.x * kAppendThreads + (int)threadIdx.x, nthreads = (int)gridDim.x * kAppendThreads;
    if (vec16)                                         // uniform
        write_rows<D, 8>(units, n, tid, nthreads);
    else
        write_rows<D, 2>(units, n, tid, nthreads);
    if (units.T < 0) return;                           // full cache: nothing is written (no block counts in)
    const int p = T % kPage, NP = a.TS / kPage, pg = T / kPage;
    // a page end: the page of every unit
    for (int u = u0; p == kPage - 1 && u < n; u += nw) {
        const int b = u / a.H, h = u % a.H;
        const int64_t row0 = ((int64_t)b * a.TS + (int64_t)pg * kPage) * a.H + h, page = units.page(u);
        const uint32_t rm = encode_page<D>(units.tail(u), D, units.x(u), lane, a.sm + row0 * D, a.code + row0 * (D / 2),
                                           a.H, a.base + page * D, nullptr);
        if (lane == 0) {
            st_dev_i32(a.rowmask + page, (int32_t)rm);
            if (pg + 1 < NP) {
                a.rowmask[page + a.H] = 0xFFFF;
                a.rowoff[page + a.H] = (int32_t)(a.cap + (int64_t)u * kPage);
            }
        }
    }
    // at a page end the last block reads every unit's rowmask: this wave's stores are
    // complete before the block counts itself in; otherwise the count only orders every
    // block's read of state[0] before the last block's write of it
    if (ONE) {
        if (p == kPage - 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    } else if (!last_block(a.state + 1, p == kPage - 1)) {
        return;
    }
    if (p == kPage - 1) {
        const RawPool pool{a.rowmask, a.rowoff, a.raw, a.cap};
        const int cnt0 = *a.cnt, rows = place_raw_rows<D, ONE ? kAppendOne : kAppendLdsUnits>(units, n, cnt0, pool);
        if (threadIdx.x == 0) {
            *a.before = cnt0;
            *a.cnt = cnt0 + rows;
        }
    }
    if (threadIdx.x == 0) {
        if (!ONE) st_dev_i32(a.state + 1, 0);
        a.state[0] = T + 1;
    }
}

// Plain bf16 cache (reference cache.py:129-146): buf[b, T, h] = x[b, h], T from device.
template <int D>
__global__ void __launch_bounds__(256) bf16_append_kernel(const uint16_t* x, int64_t sx_b, int64_t sx_h,
                                                          uint16_t* buf, const int32_t* state, int B, int H,
                                                          int TS) {
    const int lane = threadIdx.x & 63;
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= B * H) return;
    const int T = state[0];
    if (T < 0 || T >= TS) return;
    const int b = u / H, h = u % H;
    copy_row<D>(buf + (((int64_t)b * TS + T) * H + h) * D, x + b * sx_b + h * sx_h, lane);
}

__global__ void bump_kernel(int32_t* state, int TS) {
    if (state[0] < TS) state[0] += 1;
}

// Opens the page that holds token state[0] of every (sequence, head): rowmask 0xFFFF and
// rowoff = cap + (b * H + h) * 16, the (sequence, head)'s rows after the escaped-row slots.
// The page index comes from the device token count, so the caches call it when they are
// filled and after their raw pool moves, without indexing the page table on the host.
// Nothing is written for a full cache (state[0] >= TS).
__global__ void __launch_bounds__(256) open_page_kernel(int32_t* rowmask, int32_t* rowoff, const int32_t* state,
                                                        int64_t cap, int B, int H, int TS) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    const int T = state[0];
    if (u >= B * H || T < 0 || T >= TS) return;
    const int64_t page = ((int64_t)(u / H) * (TS / kPage) + T / kPage) * H + u % H;
    rowmask[page] = 0xFFFF;
    rowoff[page] = (int32_t)(cap + (int64_t)u * kPage);
}

// Paged caches: the same for sequence slots slots[0 .. n): slot s's open page is table entry
// lens[s] / 16 (when it exists), its rows at cap + (s * H + h) * 16.
__global__ void __launch_bounds__(256) open_pages_paged_kernel(int32_t* rowmask, int32_t* rowoff,
                                                               const int32_t* slots, int n, const int32_t* lens,
                                                               const int32_t* bt, int64_t bt_stride, int max_seqs,
                                                               int max_pages, int pool_pages, int64_t cap, int H) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x;
    if (u >= n * H) return;
    const int s = (int)min((uint32_t)slots[u / H], (uint32_t)(max_seqs - 1)), h = u % H;
    const int T = lens[s];
    if (T < 0 || T / kPage >= max_pages) return;
    const int64_t pidx = min((uint32_t)bt[s * bt_stride + T / kPage], (uint32_t)(pool_pages - 1));
    rowmask[pidx * H + h] = 0xFFFF;
    rowoff[pidx * H + h] = (int32_t)(cap + ((int64_t)s * H + h) * kPage);
}

// ---------------------------------------------------------------- paged append

// One token for each of n sequences held in a pool of pages. Sequence slot s (batch row i
// -> s = slots[i], or i) owns pool pages bt[s * bt_stride + pg] (clamped to the pool) and
// has lens[s] tokens, the new one included: the caller raises lens before the append, so
// the new token is token lens[s] - 1 and the kernels never write lens. Its open page is
// held in the tail area at raw rows cap + (s * H + h) * 16; when the new token fills it,
// the page is encoded into its pool page and the next table entry is opened.
struct PagedAppendArgs {
    const uint16_t* x;        // [n, H, D] (row strides sx_b, sx_h in elements)
    int64_t sx_b, sx_h;
    uint8_t* sm;
    uint8_t* code;
    uint8_t* base;
    int32_t* rowmask;
    int32_t* rowoff;
    uint16_t* raw;
    int32_t* cnt;
    int32_t* before;
    const int32_t* slots;     // [n] or nullptr
    const int32_t* lens;      // [max_seqs]
    const int32_t* bt;        // [max_seqs, bt_stride]
    int64_t bt_stride;
    int64_t cap;
    int n, H, max_seqs, max_pages, pool_pages;
};

__device__ inline int paged_slot(const PagedAppendArgs& a, int i) {
    return a.slots ? min((uint32_t)a.slots[i], (uint32_t)(a.max_seqs - 1)) : i;
}
__device__ inline int64_t paged_pidx(const PagedAppendArgs& a, int s, int pg) {
    return (int64_t)min((uint32_t)a.bt[s * a.bt_stride + pg], (uint32_t)(a.pool_pages - 1));
}
// Token index of the new token of slot s, or -1 if it does not fit.
__device__ inline int paged_new_token(const PagedAppendArgs& a, int s) {
    const int T = a.lens[s] - 1;
    return (T >= 0 && T < a.max_pages * kPage) ? T : -1;
}

// Units of a paged append: row i's head h is unit i * H + h, each at its own token
template <int D>
struct PagedUnits {
    const PagedAppendArgs& a;
    __device__ int token(int u) const { return paged_new_token(a, paged_slot(a, u / a.H)); }
    __device__ const uint16_t* x(int u) const { return a.x + (u / a.H) * a.sx_b + (u % a.H) * a.sx_h; }
    __device__ int64_t tail_row(int u) const {
        return a.cap + ((int64_t)paged_slot(a, u / a.H) * a.H + u % a.H) * kPage;
    }
    __device__ uint16_t* tail(int u) const { return a.raw + tail_row(u) * D; }
};

// The units whose page fills in this step, of the rows c0 .. c0 + 1023: listed row k's head h is
// unit k * H + h, and its page goes to pool page pidx[k].
constexpr int kFillRows = kAppendThreads;
template <int D>
struct FilledUnits {
    const PagedUnits<D>& all;
    const int* row;
    const int* pidx;
    __device__ int64_t page(int u) const { return (int64_t)pidx[u / all.a.H] * all.a.H + u % all.a.H; }
    __device__ int unit(int u) const { return row[u / all.a.H] * all.a.H + u % all.a.H; }
    __device__ const uint16_t* src_row(int u, int r) const {
        return r == kPage - 1 ? all.x(unit(u)) : all.tail(unit(u)) + r * D;
    }
};

// The pool page that row i's token fills in this step, or -1.
__device__ inline int fill_page(const PagedAppendArgs& a, int i) {
    if (i >= a.n) return -1;
    const int s = paged_slot(a, i), T = paged_new_token(a, s);
    return T >= 0 && T % kPage == kPage - 1 ? (int)paged_pidx(a, s, T / kPage) : -1;
}
// Lists the rows c0 .. c0 + 1023 of the step whose token fills a page, in order, from every
// thread's p = fill_page of row c0 + threadIdx.x; returns their number.
__device__ inline int list_fills(int c0, int p, int* row, int* pidx) {
    int nf;
    const int at = block_excl_scan(p >= 0 ? 1 : 0, nf);
    if (p >= 0) {
        row[at] = c0 + (int)threadIdx.x;
        pidx[at] = p;
    }
    __syncthreads();
    return nf;
}

// Raw-row slots and rows of the pages that the step fills, by one block; listed: the number that
// row / pidx list already, or -1.
template <int D, int LDSU>
__device__ inline void paged_place(const PagedAppendArgs& a, int* row, int* pidx, int listed) {
    const PagedUnits<D> units{a};
    int cnt0 = 0, cnt = 0;
    bool any = false;
    for (int c0 = 0; c0 < a.n; c0 += kFillRows) {
        const int nf = listed >= 0 ? listed : list_fills(c0, fill_page(a, c0 + (int)threadIdx.x), row, pidx);
        if (nf == 0) continue;                         // uniform
        if (!any) cnt0 = cnt = *a.cnt;
        any = true;
        cnt += place_raw_rows<D, LDSU>(FilledUnits<D>{units, row, pidx}, nf * a.H, cnt,
                                       RawPool{a.rowmask, a.rowoff, a.raw, a.cap});
        __syncthreads();                               // the lists are read; the counter's value too
    }
    if (any && threadIdx.x == 0) {
        *a.before = cnt0;
        *a.cnt = cnt;
    }
}

// The paged append in one launch, as append_kernel: token rows into the open pages; where
// sequences fill a page in this step, those pages encoded, the next ones opened, and their raw
// rows placed in (row, head, token) order by the last block to arrive. Every block lists the
// filling sequences from lens, which no kernel writes, 1,024 rows at a time; in a step without
// any none counts itself in. Three launches / this one, back to back, 8 KV heads of 128: 8
// sequences none of which fills a page 5.8 / 3.3 us, 16 of which one does 8.5 / 8.1, 620 of which
// 39 do 17.3 / 12.2. `arrivals`: an int32 word, zero between calls; nullptr: the raw
// rows are left to paged_place_kernel (ONE: not used).
template <int D, bool ONE>
__global__ void __launch_bounds__(kAppendThreads) paged_append_kernel(PagedAppendArgs a, int32_t* arrivals, bool vec16) {
    __shared__ int s_row[kFillRows], s_pidx[kFillRows];
    const int n = a.n * a.H, lane = threadIdx.x & 63;
    const int w0 = (int)blockIdx.x * kAppendWaves + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nw = (int)gridDim.x * kAppendWaves;
    const PagedUnits<D> units{a};
    const int tid = (int)blockIdx.x * kAppendThreads + (int)threadIdx.x, nthreads = (int)gridDim.x * kAppendThreads;
    const int p0 = fill_page(a, (int)threadIdx.x);     // its loads beside the rows'
    if (vec16)                                         // uniform
        write_rows<D, 8>(units, n, tid, nthreads);
    else
        write_rows<D, 2>(units, n, tid, nthreads);
    int nf = 0, any = 0;
    for (int c0 = 0; c0 < a.n; c0 += kFillRows) {
        if (c0 > 0) __syncthreads();                   // the lists are read
        nf = list_fills(c0, c0 > 0 ? fill_page(a, c0 + (int)threadIdx.x) : p0, s_row, s_pidx);
        any += nf;
        const FilledUnits<D> filled{units, s_row, s_pidx};
        for (int k = w0; k < nf * a.H; k += nw) {
            const int u = __builtin_amdgcn_readfirstlane(filled.unit(k)), i = u / a.H, h = u % a.H;
            const int s = paged_slot(a, i), pg = paged_new_token(a, s) / kPage;
            const int64_t page = filled.page(k), row0 = (page - h) * kPage + h;
            const uint32_t rm = encode_page<D>(units.tail(u), D, units.x(u), lane, a.sm + row0 * D,
                                               a.code + row0 * (D / 2), a.H, a.base + page * D, nullptr);
            if (lane == 0) {
                st_dev_i32(a.rowmask + page, (int32_t)rm);
                if (pg + 1 < a.max_pages) {
                    const int64_t next = paged_pidx(a, s, pg + 1) * a.H + h;
                    a.rowmask[next] = 0xFFFF;
                    a.rowoff[next] = (int32_t)units.tail_row(u);
                }
            }
        }
    }
    if (any == 0) return;                              // uniform over the grid
    if (ONE) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    } else if (arrivals == nullptr || !last_block(arrivals, true)) {
        return;
    }
    paged_place<D, ONE ? kAppendOne : kAppendLdsUnits>(a, s_row, s_pidx, a.n <= kFillRows ? nf : -1);
    if (!ONE && threadIdx.x == 0) st_dev_i32(arrivals, 0);
}

// The end of a paged append whose caller gives no arrival word: one block, after the stores.
template <int D>
__global__ void __launch_bounds__(kAppendThreads) paged_place_kernel(PagedAppendArgs a) {
    __shared__ int s_row[kFillRows], s_pidx[kFillRows];
    paged_place<D, kAppendLdsUnits>(a, s_row, s_pidx, -1);
}

// bf16 twin: pool[(page * 16 + T % 16) * H + h] = x[i, h], page = bt[s, T / 16].
template <int D>
__global__ void __launch_bounds__(256) paged_bf16_append_kernel(PagedAppendArgs a, uint16_t* buf) {
    const int lane = threadIdx.x & 63;
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= a.n * a.H) return;
    const int i = u / a.H, h = u % a.H;
    const int s = paged_slot(a, i);
    const int T = paged_new_token(a, s);
    if (T < 0) return;
    const int64_t row = paged_pidx(a, s, T / kPage) * kPage + T % kPage;
    copy_row<D>(buf + (row * a.H + h) * D, a.x + i * a.sx_b + h * a.sx_h, lane);
}

// ---------------------------------------------------------------- decode to bf16

struct DecArgs {
    CSrc c;
    uint16_t* out;            // [B, T, H, D]
    int B, T, TS, H;
    // paged: page pg of sequence b is pool page bt[b * bt_stride + pg] (clamped to pool_pages)
    const int32_t* bt = nullptr;
    int64_t bt_stride = 0;
    int64_t pool_pages = 0;
};

// One wavefront per (sequence, page, head), lane = (token r, channel group g): the page
// rebuild of the attention kernels (tile.hpp), any head dim.
template <int D>
__global__ void __launch_bounds__(256) decode_kernel(DecArgs a) {
    constexpr int R = Run<D>::R;
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int NP = a.TS / kPage;
    const int64_t u = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= (int64_t)a.B * NP * a.H) return;
    const int h = (int)(u % a.H);
    const int pg = (int)((u / a.H) % NP);
    const int b = (int)(u / ((int64_t)a.H * NP));
    if (pg * kPage >= a.T) return;
    const int t = pg * kPage + r;
    const int64_t pidx = a.bt ? (int64_t)min((uint32_t)a.bt[b * a.bt_stride + pg], (uint32_t)(a.pool_pages - 1))
                              : (int64_t)b * NP + pg;
    const int64_t page = pidx * a.H + h;
    PageBytesD<D> pb;
    load_page_d<D>(a.c, (pidx * kPage + r) * a.H + h, page, g, pb);
    const uint32_t rmask = (uint32_t)a.c.rowmask[page];
    const int32_t roff = a.c.rowoff[page];
    uint32_t v[Run<D>::V];
    rebuild_page_d<D>(a.c, pb, rmask, roff, r, g, v);
    if (t >= a.T) return;
    uint16_t* o = a.out + (((int64_t)b * a.T + t) * a.H + h) * D + g * R;
    st_words<R / 2>(o, v);
    st_words<R / 2>(o + D / 2, v + R / 2);
}

template <int D>
static void launch_decode(const DecArgs& a, int64_t n, hipStream_t stream) {
    hipLaunchKernelGGL(decode_kernel<D>, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, stream, a);
}
static void launch_decode_any(int D, const DecArgs& a, int64_t n, hipStream_t stream) {
    if (D == 64)
        launch_decode<64>(a, n, stream);
    else if (D == 256)
        launch_decode<256>(a, n, stream);
    else
        launch_decode<128>(a, n, stream);
}

}  // namespace exkv

using namespace exkv;

static int launch_status(const char* what) { return hip_status(hipGetLastError(), what); }

// The instance of kernel template K for head dim D (64, 128 or 256; checked by the caller).
#define EXKV_FOR_D(K, D) ((D) == 64 ? K<64> : (D) == 256 ? K<256> : K<128>)
#define EXKV_FOR_D2(K, D, X) ((D) == 64 ? K<64, X> : (D) == 256 ? K<256, X> : K<128, X>)

static bool rows_of_16_bytes(const void* x, int64_t sx_b, int64_t sx_h) {
    return (uintptr_t)x % 16 == 0 && sx_b % 8 == 0 && sx_h % 8 == 0;
}

// Blocks of an append over n units: one (the ONE kernels) up to kAppendOne, then a unit per wave
// up to kAppendBlocks.
static unsigned append_grid(int64_t n) {
    if (n <= kAppendOne) return 1;
    const int64_t blocks = (n + kAppendWaves - 1) / kAppendWaves;
    return (unsigned)(blocks < kAppendBlocks ? blocks : kAppendBlocks);
}

static int check_encode(const char* what, const void* src, int64_t s_b, int64_t s_pg, int64_t s_p, int64_t s_h,
                        bool pointers, int64_t cap, int64_t raw_rows, int32_t B, int32_t b0, int32_t pg0, int32_t nb,
                        int32_t npg, int32_t H, int32_t TS, int32_t D) {
    EXKV_REQUIRE(head_dim_ok(D), "%s: head dim must be 64, 128 or 256 (got %d)", what, D);
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0, "%s: TS must be a positive multiple of 16 (got %d)", what, TS);
    EXKV_REQUIRE(H > 0 && B > 0, "%s: bad H=%d or B=%d", what, H, B);
    EXKV_REQUIRE(nb >= 0 && npg >= 0 && b0 >= 0 && pg0 >= 0, "%s: negative range", what);
    EXKV_REQUIRE(b0 + nb <= B, "%s: sequences [%d, %d) outside the cache (B=%d)", what, b0, b0 + nb, B);
    EXKV_REQUIRE(pg0 + npg <= TS / kPage, "%s: pages [%d, %d) outside the cache (%d pages)", what, pg0, pg0 + npg,
                 TS / kPage);
    EXKV_REQUIRE(cap >= 0 && cap <= raw_rows, "%s: cap %lld exceeds the raw pool (%lld rows)", what, (long long)cap,
                 (long long)raw_rows);
    EXKV_REQUIRE(src && pointers, "%s: null pointer", what);
    EXKV_REQUIRE((uintptr_t)src % 4 == 0 && s_b % 2 == 0 && s_pg % 2 == 0 && s_p % 2 == 0 && s_h % 2 == 0,
                 "%s: source rows must start at even elements (4-byte aligned)", what);
    const int64_t n = (int64_t)nb * npg * H;
    EXKV_REQUIRE(n <= INT32_MAX - 1024, "%s: %lld pages x heads in one call (limit 2^31 - 1025)", what, (long long)n);
    return EXKV_OK;
}

extern "C" int exkv_encode_pages(const void* src, int64_t s_b, int64_t s_pg, int64_t s_p, int64_t s_h,
                                 void* sm, void* code, void* base, int32_t* rowmask, int32_t* rowoff, void* raw,
                                 int32_t* cnt, int32_t* before, int64_t cap, int64_t raw_rows, int32_t B,
                                 int32_t b0, int32_t pg0, int32_t nb, int32_t npg, int32_t H, int32_t TS,
                                 int32_t D, void* scan_ws, int64_t scan_ws_words, hipStream_t stream) {
    const int rc = check_encode("encode_pages", src, s_b, s_pg, s_p, s_h,
                                sm && code && base && rowmask && rowoff && raw && cnt, cap, raw_rows, B, b0, pg0, nb, npg,
                                H, TS, D);
    if (rc != EXKV_OK) return rc;
    const int64_t n = (int64_t)nb * npg * H;
    if (n == 0) return EXKV_OK;
    EXKV_REQUIRE(scan_ws == nullptr || (uintptr_t)scan_ws % 8 == 0, "encode_pages: scan workspace must be 8-byte aligned");
    EncArgs a{(const uint16_t*)src, s_b, s_pg, s_p, s_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base,
              rowmask, rowoff, (uint16_t*)raw, cnt, before, cap, b0, pg0, nb, npg, H, TS};
    a.D = D;
    launch_encode(a, n, (uint64_t*)scan_ws, scan_ws_words, nullptr, stream);
    return launch_status("encode_pages");
}

template <int D>
static void launch_store_raw(const EncArgs& a, int64_t n, hipStream_t stream) {
    const unsigned grid = (unsigned)((n + 4 * kStoreUnits - 1) / (4 * kStoreUnits));
    auto k = rows_of_16_bytes(a) ? store_raw_kernel<true, D> : store_raw_kernel<false, D>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, stream, a, (int)n);
}

extern "C" int exkv_store_raw_rows(const void* src, int64_t s_b, int64_t s_pg, int64_t s_p, int64_t s_h,
                                   const int32_t* rowmask, const int32_t* rowoff, void* raw, int64_t cap,
                                   int64_t raw_rows, int32_t B, int32_t b0, int32_t pg0, int32_t nb, int32_t npg,
                                   int32_t H, int32_t TS, int32_t D, hipStream_t stream) {
    const int rc = check_encode("store_raw_rows", src, s_b, s_pg, s_p, s_h, rowmask && rowoff && raw, cap, raw_rows, B,
                                b0, pg0, nb, npg, H, TS, D);
    if (rc != EXKV_OK) return rc;
    const int64_t n = (int64_t)nb * npg * H;
    if (n == 0) return EXKV_OK;
    EncArgs a{(const uint16_t*)src, s_b, s_pg, s_p, s_h, nullptr, nullptr, nullptr, const_cast<int32_t*>(rowmask),
              const_cast<int32_t*>(rowoff), (uint16_t*)raw, nullptr, nullptr, cap, b0, pg0, nb, npg, H, TS};
    if (D == 64)
        launch_store_raw<64>(a, n, stream);
    else if (D == 256)
        launch_store_raw<256>(a, n, stream);
    else
        launch_store_raw<128>(a, n, stream);
    return launch_status("store_raw_rows");
}

// Pages of nb source sequences x npg pages into arbitrary pages of B x TS caches read as a
// list of B * TS / 16 pages: page pg of source sequence bi goes to page dst_pages[bi *
// dst_stride + pg]. Same kernels, raw-slot order (unit order) and bytes as
// exkv_encode_pages.
extern "C" int exkv_encode_pages_paged(const void* src, int64_t s_b, int64_t s_pg, int64_t s_p, int64_t s_h,
                                       void* sm, void* code, void* base, int32_t* rowmask, int32_t* rowoff,
                                       void* raw, int32_t* cnt, int32_t* before, int64_t cap, int64_t raw_rows,
                                       int32_t B, const int32_t* dst_pages, int64_t dst_stride, int32_t nb,
                                       int32_t npg, int32_t H, int32_t TS, int32_t D, void* scan_ws,
                                       int64_t scan_ws_words, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "encode_pages_paged: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0, "encode_pages_paged: TS must be a positive multiple of 16 (got %d)", TS);
    EXKV_REQUIRE(H > 0 && B > 0, "encode_pages_paged: bad H=%d or B=%d", H, B);
    EXKV_REQUIRE(nb >= 0 && npg >= 0, "encode_pages_paged: negative range");
    EXKV_REQUIRE(dst_pages && dst_stride >= npg, "encode_pages_paged: need a page table of >= %d columns", npg);
    EXKV_REQUIRE(cap >= 0 && cap <= raw_rows, "encode_pages_paged: cap %lld exceeds the raw pool (%lld rows)",
                 (long long)cap, (long long)raw_rows);
    EXKV_REQUIRE(src && sm && code && base && rowmask && rowoff && raw && cnt, "encode_pages_paged: null pointer");
    EXKV_REQUIRE((uintptr_t)src % 4 == 0 && s_b % 2 == 0 && s_pg % 2 == 0 && s_p % 2 == 0 && s_h % 2 == 0,
                 "encode_pages_paged: source rows must start at even elements (4-byte aligned)");
    const int64_t n = (int64_t)nb * npg * H;
    if (n == 0) return EXKV_OK;
    EXKV_REQUIRE(n <= INT32_MAX - 1024, "encode_pages_paged: %lld pages x heads in one call (limit 2^31 - 1025)",
                 (long long)n);
    EncArgs a{(const uint16_t*)src, s_b, s_pg, s_p, s_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base,
              rowmask, rowoff, (uint16_t*)raw, cnt, before, cap, 0, 0, nb, npg, H, TS};
    a.dst_pages = dst_pages;
    a.dst_stride = dst_stride;
    a.all_pages = (int64_t)B * (TS / kPage);
    a.D = D;
    EXKV_REQUIRE(scan_ws == nullptr || (uintptr_t)scan_ws % 8 == 0,
                 "encode_pages_paged: scan workspace must be 8-byte aligned");
    launch_encode(a, n, (uint64_t*)scan_ws, scan_ws_words, nullptr, stream);
    return launch_status("encode_pages_paged");
}

// A prompt into sequence slot b in two launches (one below a page of tokens): its full pages as
// exkv_encode_pages encodes them, its last rows into the slot's open page, page T / 16 of every
// sequence opened (exkv_cache_open_page), state[0] = T.
static int prefill_slot(const char* what, EncArgs& a, PrefillEnd& e, int64_t s_t, int64_t s_h, int32_t T, int64_t slot,
                        int64_t slots, int64_t raw_rows, int32_t D, void* scan_ws, int64_t scan_ws_words, int32_t* host,
                        int32_t tag, int32_t* arrivals, hipStream_t stream) {
    const int64_t tail_end = a.cap + slots * a.H * kPage;
    EXKV_REQUIRE(a.cap >= 0 && tail_end <= raw_rows && tail_end <= INT32_MAX,
                 "%s: raw pool (%lld rows) smaller than cap + open-page rows", what, (long long)raw_rows);
    EXKV_REQUIRE(a.src && a.sm && a.code && a.base && a.rowmask && a.rowoff && a.raw && a.cnt,
                 "%s: null pointer", what);
    EXKV_REQUIRE(s_t >= 0 && s_h >= 0, "%s: negative source strides", what);
    const int64_t n = (int64_t)a.npg * a.H;
    EXKV_REQUIRE(n == 0 || ((uintptr_t)a.src % 4 == 0 && s_t % 2 == 0 && s_h % 2 == 0),
                 "%s: source rows must start at even elements (4-byte aligned)", what);
    EXKV_REQUIRE(n <= INT32_MAX - 1024, "%s: %lld pages x heads in one call (limit 2^31 - 1025)", what, (long long)n);
    EXKV_REQUIRE(scan_ws == nullptr || (uintptr_t)scan_ws % 8 == 0, "%s: scan workspace must be 8-byte aligned", what);
    if (host != nullptr) {
        EXKV_REQUIRE(arrivals, "%s: null pointer", what);
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        const hipError_t st = hipStreamIsCapturing(stream, &capturing);
        if (st != hipSuccess) return hip_status(st, what);
        EXKV_REQUIRE(capturing == hipStreamCaptureStatusNone, "%s: the stream is being captured", what);
    }
    a.D = D;
    e.host = host;
    e.tag = tag;
    e.arrivals = arrivals;
    e.tail = a.src + (int64_t)a.npg * kPage * s_t;
    e.s_t = s_t;
    e.s_h = s_h;
    e.rows = T % kPage;
    e.tail0 = a.cap + slot * a.H * kPage;
    e.T = T;
    launch_encode(a, n, (uint64_t*)scan_ws, scan_ws_words, &e, stream);
    const int rc = launch_status(what);
    return rc != EXKV_OK || host == nullptr ? rc : wait_for_tag(what, host, tag, stream);
}

extern "C" int exkv_prefill_slot(const void* src, int64_t s_t, int64_t s_h, int32_t T, void* sm, void* code, void* base,
                                 int32_t* rowmask, int32_t* rowoff, void* raw, int32_t* cnt, int32_t* before,
                                 int32_t* state, int64_t cap, int64_t raw_rows, int32_t B, int32_t b, int32_t H,
                                 int32_t TS, int32_t D, void* scan_ws, int64_t scan_ws_words, int32_t* host,
                                 int32_t tag, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "prefill_slot: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0 && B > 0 && H > 0, "prefill_slot: bad shape B=%d H=%d TS=%d", B, H, TS);
    EXKV_REQUIRE(b >= 0 && b < B && T >= 0 && T <= TS, "prefill_slot: %d tokens into slot %d outside the cache", T, b);
    EXKV_REQUIRE(state, "prefill_slot: null pointer");
    EncArgs a{(const uint16_t*)src, 0, kPage * s_t, s_t, s_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base,
              rowmask, rowoff, (uint16_t*)raw, cnt, before, cap, b, 0, 1, T / kPage, H, TS};
    PrefillEnd e;
    e.state = state;
    e.B = B;
    e.open_pages = TS / kPage;
    return prefill_slot("prefill_slot", a, e, s_t, s_h, T, b, B, raw_rows, D, scan_ws, scan_ws_words, host, tag, state + 1,
                        stream);
}

// The same into slot `slot` of a paged cache: its page p is pool page table[p] (entries clamped
// to the pool), and page T / 16 is opened where the table has it.
extern "C" int exkv_prefill_slot_paged(const void* src, int64_t s_t, int64_t s_h, int32_t T, void* sm, void* code,
                                       void* base, int32_t* rowmask, int32_t* rowoff, void* raw, int32_t* cnt,
                                       int32_t* before, int32_t* arrivals, int64_t cap, int64_t raw_rows,
                                       const int32_t* table, int32_t slot, int32_t max_seqs, int32_t max_pages,
                                       int32_t pool_pages, int32_t H, int32_t D, void* scan_ws, int64_t scan_ws_words,
                                       int32_t* host, int32_t tag, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "prefill_slot_paged: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(H > 0 && max_seqs > 0 && max_pages > 0 && pool_pages > 0, "prefill_slot_paged: bad shape");
    EXKV_REQUIRE(slot >= 0 && slot < max_seqs && T >= 0 && T <= (int64_t)max_pages * kPage,
                 "prefill_slot_paged: %d tokens into slot %d outside the cache", T, slot);
    EXKV_REQUIRE(table, "prefill_slot_paged: null pointer");
    EncArgs a{(const uint16_t*)src, 0, kPage * s_t, s_t, s_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base,
              rowmask, rowoff, (uint16_t*)raw, cnt, before, cap, 0, 0, 1, T / kPage, H, kPage};
    a.dst_pages = table;
    a.dst_stride = max_pages;
    a.all_pages = pool_pages;
    PrefillEnd e;
    e.open_pages = max_pages;
    e.table = table;
    e.pool_pages = pool_pages;
    return prefill_slot("prefill_slot_paged", a, e, s_t, s_h, T, slot, max_seqs, raw_rows, D, scan_ws, scan_ws_words, host,
                        tag, arrivals, stream);
}

extern "C" int exkv_cache_append(const void* x, int64_t sx_b, int64_t sx_h, void* sm, void* code, void* base,
                                 int32_t* rowmask, int32_t* rowoff, void* raw, int32_t* cnt, int32_t* before,
                                 int32_t* state, int64_t cap, int64_t raw_rows, int32_t B, int32_t H,
                                 int32_t TS, int32_t D, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "append: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0 && B > 0 && H > 0, "append: bad shape B=%d H=%d TS=%d", B, H, TS);
    EXKV_REQUIRE(cap >= 0 && cap + (int64_t)B * H * kPage <= raw_rows,
                 "append: raw pool (%lld rows) smaller than cap + tail area", (long long)raw_rows);
    EXKV_REQUIRE(x && sm && code && base && rowmask && rowoff && raw && cnt && before && state,
                 "append: null pointer");
    EXKV_REQUIRE((uintptr_t)x % 4 == 0 && sx_b % 2 == 0 && sx_h % 2 == 0,
                 "append: token rows must start at even elements (4-byte aligned)");
    AppendArgs a{(const uint16_t*)x, sx_b, sx_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base, rowmask, rowoff,
                 (uint16_t*)raw, cnt, before, state, cap, B, H, TS};
    const unsigned grid = append_grid((int64_t)B * H);
    auto k = grid == 1 ? EXKV_FOR_D2(append_kernel, D, true) : EXKV_FOR_D2(append_kernel, D, false);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kAppendThreads), 0, stream, a, rows_of_16_bytes(x, sx_b, sx_h));
    return launch_status("cache_append");
}

extern "C" int exkv_bf16_append(const void* x, int64_t sx_b, int64_t sx_h, void* buf, int32_t* state,
                                int32_t B, int32_t H, int32_t TS, int32_t D, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "bf16_append: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(B > 0 && H > 0 && TS > 0, "bf16_append: bad shape");
    EXKV_REQUIRE(x && buf && state, "bf16_append: null pointer");
    hipLaunchKernelGGL(EXKV_FOR_D(bf16_append_kernel, D), dim3((unsigned)((B * H + 3) / 4)), dim3(256), 0, stream,
                       (const uint16_t*)x, sx_b, sx_h, (uint16_t*)buf, (const int32_t*)state, B, H, TS);
    hipLaunchKernelGGL(bump_kernel, dim3(1), dim3(1), 0, stream, state, TS);
    return launch_status("bf16_append");
}

extern "C" int exkv_cache_open_page(int32_t* rowmask, int32_t* rowoff, const int32_t* state, int64_t cap,
                                    int64_t raw_rows, int32_t B, int32_t H, int32_t TS, hipStream_t stream) {
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0 && B > 0 && H > 0, "open_page: bad shape B=%d H=%d TS=%d", B, H, TS);
    EXKV_REQUIRE(cap >= 0 && cap + (int64_t)B * H * kPage <= raw_rows && cap + (int64_t)B * H * kPage <= INT32_MAX,
                 "open_page: raw pool (%lld rows) smaller than cap + tail area", (long long)raw_rows);
    EXKV_REQUIRE(rowmask && rowoff && state, "open_page: null pointer");
    hipLaunchKernelGGL(open_page_kernel, dim3((unsigned)((B * H + 255) / 256)), dim3(256), 0, stream, rowmask,
                       rowoff, state, cap, B, H, TS);
    return launch_status("cache_open_page");
}

extern "C" int exkv_cache_open_pages_paged(int32_t* rowmask, int32_t* rowoff, const int32_t* slots, int32_t n,
                                           const int32_t* lens, const int32_t* block_table, int64_t bt_stride,
                                           int32_t max_seqs, int32_t max_pages, int32_t pool_pages, int64_t cap,
                                           int64_t raw_rows, int32_t H, hipStream_t stream) {
    EXKV_REQUIRE(n >= 0 && n <= max_seqs && H > 0 && max_pages > 0 && bt_stride >= max_pages && pool_pages > 0,
                 "open_pages_paged: bad shape n=%d H=%d max_seqs=%d max_pages=%d", n, H, max_seqs, max_pages);
    EXKV_REQUIRE(cap >= 0 && cap + (int64_t)max_seqs * H * kPage <= raw_rows &&
                     cap + (int64_t)max_seqs * H * kPage <= INT32_MAX,
                 "open_pages_paged: raw pool (%lld rows) smaller than cap + tail area", (long long)raw_rows);
    EXKV_REQUIRE(rowmask && rowoff && lens && block_table && (slots || n == 0), "open_pages_paged: null pointer");
    if (n == 0) return EXKV_OK;
    hipLaunchKernelGGL(open_pages_paged_kernel, dim3((unsigned)((n * H + 255) / 256)), dim3(256), 0, stream,
                       rowmask, rowoff, slots, n, lens, block_table, bt_stride, max_seqs, max_pages, pool_pages, cap,
                       H);
    return launch_status("cache_open_pages_paged");
}

static int check_paged_append(const char* what, int32_t n, int32_t H, int32_t D, int32_t max_seqs,
                              int32_t max_pages, int64_t bt_stride, int32_t pool_pages) {
    EXKV_REQUIRE(head_dim_ok(D), "%s: head dim must be 64, 128 or 256 (got %d)", what, D);
    EXKV_REQUIRE(n >= 0 && H > 0 && max_seqs > 0 && n <= max_seqs, "%s: bad shape n=%d H=%d max_seqs=%d", what, n,
                 H, max_seqs);
    EXKV_REQUIRE(max_pages > 0 && bt_stride >= max_pages && pool_pages > 0,
                 "%s: bad page table (max_pages=%d stride=%lld pool=%d)", what, max_pages, (long long)bt_stride,
                 pool_pages);
    return EXKV_OK;
}

static int append_paged(const char* what, const PagedAppendArgs& a, int64_t raw_rows, int32_t D, int32_t* arrivals,
                        hipStream_t stream) {
    const int rc = check_paged_append(what, a.n, a.H, D, a.max_seqs, a.max_pages, a.bt_stride, a.pool_pages);
    if (rc != EXKV_OK) return rc;
    EXKV_REQUIRE(a.cap >= 0 && a.cap + (int64_t)a.max_seqs * a.H * kPage <= raw_rows,
                 "%s: raw pool (%lld rows) smaller than cap + tail area", what, (long long)raw_rows);
    EXKV_REQUIRE(a.x && a.sm && a.code && a.base && a.rowmask && a.rowoff && a.raw && a.cnt && a.before && a.lens && a.bt,
                 "%s: null pointer", what);
    EXKV_REQUIRE((uintptr_t)a.x % 4 == 0 && a.sx_b % 2 == 0 && a.sx_h % 2 == 0,
                 "%s: token rows must start at even elements (4-byte aligned)", what);
    if (a.n == 0) return EXKV_OK;
    const unsigned grid = append_grid((int64_t)a.n * a.H);
    auto k = grid == 1 ? EXKV_FOR_D2(paged_append_kernel, D, true) : EXKV_FOR_D2(paged_append_kernel, D, false);
    hipLaunchKernelGGL(k, dim3(grid), dim3(kAppendThreads), 0, stream, a, arrivals,
                       rows_of_16_bytes(a.x, a.sx_b, a.sx_h));
    if (grid > 1 && arrivals == nullptr)
        hipLaunchKernelGGL(EXKV_FOR_D(paged_place_kernel, D), dim3(1), dim3(kAppendThreads), 0, stream, a);
    return launch_status(what);
}

extern "C" int exkv_cache_append_paged(const void* x, int64_t sx_b, int64_t sx_h, void* sm, void* code, void* base,
                                       int32_t* rowmask, int32_t* rowoff, void* raw, int32_t* cnt, int32_t* before,
                                       int64_t cap, int64_t raw_rows, const int32_t* slots, const int32_t* lens,
                                       const int32_t* block_table, int64_t bt_stride, int32_t n, int32_t H,
                                       int32_t max_seqs, int32_t max_pages, int32_t pool_pages, int32_t D,
                                       hipStream_t stream) {
    const PagedAppendArgs a{(const uint16_t*)x, sx_b, sx_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base, rowmask,
                            rowoff, (uint16_t*)raw, cnt, before, slots, lens, block_table, bt_stride, cap, n, H,
                            max_seqs, max_pages, pool_pages};
    return append_paged("append_paged", a, raw_rows, D, nullptr, stream);
}

extern "C" int exkv_cache_append_paged_counted(const void* x, int64_t sx_b, int64_t sx_h, void* sm, void* code,
                                               void* base, int32_t* rowmask, int32_t* rowoff, void* raw, int32_t* cnt,
                                               int32_t* before, int32_t* arrivals, int64_t cap, int64_t raw_rows,
                                               const int32_t* slots, const int32_t* lens, const int32_t* block_table,
                                               int64_t bt_stride, int32_t n, int32_t H, int32_t max_seqs,
                                               int32_t max_pages, int32_t pool_pages, int32_t D, hipStream_t stream) {
    EXKV_REQUIRE(arrivals, "append_paged: null pointer");
    const PagedAppendArgs a{(const uint16_t*)x, sx_b, sx_h, (uint8_t*)sm, (uint8_t*)code, (uint8_t*)base, rowmask,
                            rowoff, (uint16_t*)raw, cnt, before, slots, lens, block_table, bt_stride, cap, n, H,
                            max_seqs, max_pages, pool_pages};
    return append_paged("append_paged", a, raw_rows, D, arrivals, stream);
}

extern "C" int exkv_bf16_append_paged(const void* x, int64_t sx_b, int64_t sx_h, void* buf, const int32_t* slots,
                                      const int32_t* lens, const int32_t* block_table, int64_t bt_stride, int32_t n,
                                      int32_t H, int32_t max_seqs, int32_t max_pages, int32_t pool_pages, int32_t D,
                                      hipStream_t stream) {
    const int rc = check_paged_append("bf16_append_paged", n, H, D, max_seqs, max_pages, bt_stride, pool_pages);
    if (rc != EXKV_OK) return rc;
    EXKV_REQUIRE(x && buf && lens && block_table, "bf16_append_paged: null pointer");
    if (n == 0) return EXKV_OK;
    PagedAppendArgs a{(const uint16_t*)x, sx_b, sx_h, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                      nullptr, nullptr, slots, lens, block_table, bt_stride, 0, n, H, max_seqs, max_pages,
                      pool_pages};
    hipLaunchKernelGGL(EXKV_FOR_D(paged_bf16_append_kernel, D), dim3((unsigned)((n * H + 3) / 4)), dim3(256), 0,
                       stream, a, (uint16_t*)buf);
    return launch_status("bf16_append_paged");
}

extern "C" int exkv_decode_to_bf16_paged(const void* sm, const void* code, const void* base,
                                         const int32_t* rowmask, const int32_t* rowoff, const void* raw,
                                         int64_t raw_rows, int64_t pool_pages, const int32_t* block_table,
                                         int64_t bt_stride, void* out, int32_t B, int32_t T, int32_t H, int32_t D,
                                         hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "decode_to_bf16_paged: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(B > 0 && H > 0 && bt_stride > 0 && pool_pages > 0, "decode_to_bf16_paged: bad shape");
    EXKV_REQUIRE(T >= 0 && T <= bt_stride * kPage, "decode_to_bf16_paged: T=%d exceeds the table's %lld pages", T,
                 (long long)bt_stride);
    EXKV_REQUIRE(raw_rows > 0, "decode_to_bf16_paged: empty raw pool");
    EXKV_REQUIRE(sm && code && base && rowmask && rowoff && raw && out && block_table,
                 "decode_to_bf16_paged: null pointer");
    if (T == 0) return EXKV_OK;
    const int TS = (T + kPage - 1) / kPage * kPage;     // pages the tokens touch
    DecArgs a{CSrc{(const uint8_t*)sm, (const uint8_t*)code, (const uint8_t*)base, rowmask, rowoff,
                   (const uint16_t*)raw, raw_rows},
              (uint16_t*)out, B, T, TS, H};
    a.bt = block_table;
    a.bt_stride = bt_stride;
    a.pool_pages = pool_pages;
    launch_decode_any(D, a, (int64_t)B * (TS / kPage) * H, stream);
    return launch_status("decode_to_bf16_paged");
}

extern "C" int exkv_decode_to_bf16(const void* sm, const void* code, const void* base, const int32_t* rowmask,
                                   const int32_t* rowoff, const void* raw, int64_t raw_rows, void* out,
                                   int32_t B, int32_t T, int32_t TS, int32_t H, int32_t D, hipStream_t stream) {
    EXKV_REQUIRE(head_dim_ok(D), "decode_to_bf16: head dim must be 64, 128 or 256 (got %d)", D);
    EXKV_REQUIRE(TS > 0 && TS % kPage == 0 && B > 0 && H > 0, "decode_to_bf16: bad shape");
    EXKV_REQUIRE(T >= 0 && T <= TS, "decode_to_bf16: T=%d outside [0, TS=%d]", T, TS);
    EXKV_REQUIRE(raw_rows > 0, "decode_to_bf16: empty raw pool");
    EXKV_REQUIRE(sm && code && base && rowmask && rowoff && raw && out, "decode_to_bf16: null pointer");
    if (T == 0) return EXKV_OK;
    DecArgs a{CSrc{(const uint8_t*)sm, (const uint8_t*)code, (const uint8_t*)base, rowmask, rowoff,
                   (const uint16_t*)raw, raw_rows},
              (uint16_t*)out, B, T, TS, H};
    launch_decode_any(D, a, (int64_t)B * (TS / kPage) * H, stream);
    return launch_status("decode_to_bf16");
}

namespace exkv {
hipError_t fetch_errors_encode(uint32_t* out, int first, int clear, hipStream_t stream) {
    return fetch_file_errors(out, first, clear, stream);
}
}  // namespace exkv
