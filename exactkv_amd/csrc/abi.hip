// C-ABI plumbing: version, error messages, the split planner.
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <algorithm>

#include "common.hpp"
#include "../../include/exactkv.h"

namespace exkv {

static thread_local char g_err[512];

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int hip_status(hipError_t e, const char* where) {
    if (e == hipSuccess) return EXKV_OK;
    set_error("%s: HIP error %d (%s)", where, (int)e, hipGetErrorString(e));
    return EXKV_E_HIP;
}

}  // namespace exkv

extern "C" int exkv_abi_version(void) { return 4; }

extern "C" int exkv_error_bits(uint32_t* out, int32_t clear, hipStream_t stream) {
    EXKV_REQUIRE(out, "error_bits: null output");
    hipError_t e = exkv::fetch_errors_attention(out, 1, clear, stream);
    if (e == hipSuccess) e = exkv::fetch_errors_encode(out, 0, clear, stream);
    if (e == hipSuccess) e = exkv::fetch_errors_wire(out, 0, clear, stream);
    return exkv::hip_status(e, "error_bits");
}

extern "C" const char* exkv_last_error(void) { return exkv::g_err; }

// Split plan for MI355X, over units = B * (Hkv / HW) * query-head groups, where a workgroup
// covers HW = min(gcd(Hkv, 8), 4) KV heads and `slots` workgroups run side by side (256: one
// per CU, by its LDS ring; the head-dim-256 kernel two per CU). Plays the role of the
// reference's choose_split (kernels.py:273-277), which targets 512 programs.
//
// A call's time follows the rounds its grid needs, R = ceil(r), r = units * ns / slots, and the
// pages that one wavefront walks per workgroup, j = ceil(split pages / page phases). In pages
// (2.05 us at head dim 128 with every CU streaming, 6.4 TB/s; 0.85 of that where the last
// round leaves CUs idle, when the page's compute bounds it): every round costs j pages and
// `ramp` more (a workgroup's first page's latency and its epilogue, 6 us), and the last
// workgroups end spread over a sixteenth of their own time:
//   cost = R ramp + j (R - 1 + max(last round's share, 0.85)) + (ramp + j) / 16.
// Over a sweep of 43 shapes (B 1 to 220, 1 to 440 units, T 512 to 32763; profiles/plan_sweep.md) it
// is 0.91 to 1.13 of the time of the plans it chooses from 30 us on, and the plan is within 2% of
// the best one timed but for one shape (10%): 24 x 4093 at 32q/8kv, 5 splits x 832 (240
// workgroups) 56.5 us, 6 x 704 (288: two rounds, the second nearly empty) 82.8, 10 x 416 59.7. For
// each R the best plan is the most splits that fit R rounds, so eight of them are compared, and of
// equal ones the first (fewer rounds, more splits) is taken. Rounding the split count up instead of
// down costs 1.3 to 1.6 times the time wherever the unit count does not divide 256 (same calls,
// split count up / down: 3 x 4093 21.2 / 15.6 us, 6 x 8192 50.6 / 31.8, 12 x 4093 45.5 / 31.6,
// 40 x 2048 64.1 / 46.7; head dim 64 24 x 4093 50.1 / 35.3; head dim 256 9 x 4093 80.7 / 52.7).
// Short splits cost little: a wavefront's pages follow one another at about one memory round
// trip each, so few units are served best by many splits, down to min_split tokens (16 by
// default, one page; measured with one round, 64- / 32- / 16-token splits: a 1024-token window
// of one B1 x 128K sequence 14.2 / 11.1 / 9.6 us).
static double plan_cost(int64_t units, int64_t ns, int64_t pages, int64_t slots, int nph, double ramp) {
    const double j = (double)(((pages + ns - 1) / ns + nph - 1) / nph);
    const double full = (double)((units * ns + slots - 1) / slots - 1);            // rounds before the last
    const double last = (double)(units * ns) / (double)slots - full;
    return (full + 1.0) * ramp + j * (full + std::max(last, 0.85)) + (ramp + j) / 16.0;
}

// The fewest splits with at least two rounds and the last one at least 95% full, else the
// fullest: the plan of grids larger than the GPU (the second round's workgroups start as the
// first ones end, which staggers the tail; measured at B256 x 4352, 1/2/4/8 splits:
// 610/601/614/636 us; B620: 2 splits 1454 us, 4 splits 1490 us), unless plan_cost finds one
// more than a sixteenth (about its error) cheaper, as it does for short contexts (B220 x 1000:
// 4 x 256 150.3 us, 1 x 1008 122.0).
static int64_t full_rounds(int64_t units, int64_t slots) {
    int64_t ns = 1;
    double best = -1.0;
    for (int64_t n = 1; n <= 16; ++n) {
        const double rounds = (double)(units * n) / slots;
        if (rounds < 2.0) continue;
        const double full = rounds / (double)(int64_t)(rounds + 0.999999);
        if (full > best) {
            best = full;
            ns = n;
        }
        if (full >= 0.95) break;
    }
    return ns;
}

// The plan, for workgroups of nph page phases; `most`: the splits whose partials fit the
// no-alloc entry point's scratch, which bounds what the cost model is asked. The plans of
// full_rounds, and of head dim 64 with odd KV heads, are not bounded by it: for many long sequences
// that entry point needs its caller's own, smaller plan (129 x 8192 at 32q/8kv: 16 splits, of
// which 15 fit).
static void plan_core(int64_t units, int32_t T, int64_t slots, int32_t min_split, int nph, double ramp, int64_t most,
                      int32_t* nsplit, int32_t* split_len) {
    const int64_t pages = ((int64_t)T + exkv::kPage - 1) / exkv::kPage;
    const int64_t cap = std::max<int64_t>(1, ((int64_t)T + min_split - 1) / min_split);
    const int64_t first = (units + slots - 1) / slots;
    // no split is shorter than min_split (or all of T): ceil(T / cap) may be
    const int64_t least = std::min(pages, ((int64_t)min_split + exkv::kPage - 1) / exkv::kPage) * exkv::kPage;
    const auto plan = [&](int64_t sl) {
        sl = std::max(sl, least);
        *split_len = (int32_t)sl;
        *nsplit = (int32_t)(((int64_t)T + sl - 1) / sl);
    };
    int64_t ns = 1;
    double cost = 0.0;
    for (int64_t r = first; r < first + 8; ++r) {
        const int64_t n = std::min(std::max<int64_t>(1, slots * r / units), std::min(cap, most));
        const double c = plan_cost(units, n, pages, slots, nph, ramp);
        if (r == first || c < cost) {
            cost = c;
            ns = n;
        }
        if (n == cap || n == most) break;
    }
    if (units >= slots) {
        const int64_t n = std::min(full_rounds(units, slots), cap);
        if (plan_cost(units, n, pages, slots, nph, ramp) <= cost * 17.0 / 16.0) {
            const int64_t sl = ((int64_t)T + n - 1) / n;
            plan(sl <= exkv::kPage ? exkv::kPage : (sl + 31) / 32 * 32);
            return;
        }
    }
    plan((pages + ns - 1) / ns * exkv::kPage);
}

// KV heads (or pairs of them) per workgroup: min(gcd(n, 8), 4)
static int heads_per_block(int n) {
    int hw = n, m = 8;
    while (m) {
        const int t = hw % m;
        hw = m;
        m = t;
    }
    return hw > 4 ? 4 : hw;
}
static int64_t scratch_splits(int64_t B, int64_t Hq, int64_t D) {
    return std::max<int64_t>(1, exkv_noalloc_scratch_bytes() / ((D + 2) * 4) / (B * Hq));
}
constexpr int kComputeWaves = 8;
constexpr double kRamp = 2.9, kRampD256 = 5.4;         // head dim 128 and pairs; 256 (2.1 us a page, 11 us a workgroup)

extern "C" int exkv_plan_splits(int32_t B, int32_t Hkv, int32_t Hq, int32_t T, int32_t target_blocks,
                                int32_t min_split, int32_t* nsplit, int32_t* split_len) {
    EXKV_REQUIRE(B > 0 && Hkv > 0 && Hq > 0 && Hq % Hkv == 0 && T > 0, "plan_splits: bad arguments");
    EXKV_REQUIRE(nsplit && split_len, "plan_splits: null output");
    if (target_blocks <= 0) target_blocks = 256;
    if (min_split <= 0) min_split = exkv::kPage;
    const int hw = heads_per_block(Hkv);
    plan_core((int64_t)B * (Hkv / hw) * ((Hq / Hkv + 15) / 16), T, target_blocks, min_split, kComputeWaves / hw, kRamp,
              scratch_splits(B, Hq, exkv::kD), nsplit, split_len);
    return EXKV_OK;
}

// Split plan per head dim. 128: the plan of exkv_plan_splits with its defaults. 64 with an
// even number of KV heads runs the head-dim-128 kernel structure over pairs of heads
// (virtual heads of 128 bytes per row): the same plan over Hkv / 2 virtual heads, a
// workgroup covering min(gcd(Hkv / 2, 8), 4) of them. Otherwise (256, or 64 with an odd
// count) the generic kernel, whose workgroups cover one KV head and one group of 16 query
// heads: rounds are counted in 512 workgroups, two per CU (the GPU holds three at head dim
// 64, two at 256, by their LDS rings); with fewer units than that, head dim 64 fills all
// three slots of every CU (768 workgroups). Measured at the c2a shape (B8 x 8192, 32q/8kv,
// split kernel): at 256, 8 splits 88.3 us against 153.1 / 95.0 for 4 / 16.
extern "C" int exkv_plan_splits_hd(int32_t B, int32_t Hkv, int32_t Hq, int32_t T, int32_t D, int32_t* nsplit,
                                   int32_t* split_len) {
    EXKV_REQUIRE(exkv::head_dim_ok(D), "plan_splits_hd: head dim must be 64, 128 or 256 (got %d)", D);
    if (D == 128) return exkv_plan_splits(B, Hkv, Hq, T, 0, 0, nsplit, split_len);
    EXKV_REQUIRE(B > 0 && Hkv > 0 && Hq > 0 && Hq % Hkv == 0 && T > 0, "plan_splits_hd: bad arguments");
    EXKV_REQUIRE(nsplit && split_len, "plan_splits_hd: null output");
    if (D == 64 && Hkv % 2 == 0) {
        const int hw = heads_per_block(Hkv / 2);
        plan_core((int64_t)B * (Hkv / 2 / hw) * ((Hq / Hkv + 15) / 16), T, 256, exkv::kPage, kComputeWaves / hw, kRamp,
                  scratch_splits(B, Hq, D), nsplit, split_len);
        return EXKV_OK;
    }
    const int64_t units = (int64_t)B * Hkv * ((Hq / Hkv + 15) / 16);
    if (D == 256) {
        // down to a page per phase: 1 x 1000 at 32q/8kv 32 x 32 11.8 us, 16 x 64 13.3; 1 x 4093 at
        // 16q/2kv 128 x 32 11.3, 64 x 64 13.3, 256 x 16 12.5
        plan_core(units, T, 512, 32, 2, kRampD256, scratch_splits(B, Hq, D), nsplit, split_len);
        return EXKV_OK;
    }
    const int64_t slots = units < 512 ? 768 : 512, cap = std::max<int64_t>(1, ((int64_t)T + 63) / 64);
    const int64_t ns = std::min(units < slots ? (slots + units - 1) / units : full_rounds(units, slots), cap);
    *split_len = (int32_t)std::max<int64_t>(exkv::kPage, (((int64_t)T + ns - 1) / ns + 31) / 32 * 32);
    *nsplit = (int32_t)(((int64_t)T + *split_len - 1) / *split_len);
    return EXKV_OK;
}
