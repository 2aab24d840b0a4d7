// tsm_nucleus.h - rows without top-k whose nucleus holds more than 1024
// candidates (the cutoff set, sampler.rs:195-208): the reference's sequential
// f32 folds reproduced exactly, over value bins.
//
// The reference folds best first, in f32: total = sum of p_j; acc += p_j /
// total until acc >= top_p (sampler.rs:238-245); mass = the kept prefix's sum
// (sampler.rs:142); r = u * mass, r -= p_j until r <= 0 (sampler.rs:143-149).
// While a fold's value x stays in one binade [2^e, 2^(e+1)), the step x + tau
// rounds tau to the grid 2^(e-23): it adds RN_e(tau) grid units whatever the
// order of the terms, unless tau lies exactly halfway between two grid points
// (then the result's parity decides).  A subtraction rounds on the grid of its
// result, the binade below when x is a power of two.  So over a value bin (a
// range of values: a contiguous stretch of the sorted list) a fold advances by
// the bin's sum of RN_e terms, as long as it neither leaves the binade nor
// meets such a tie nor reaches its decision inside the bin.
//
// A re-read pass computes, per bin, the sums for the one or two grids the bin
// can see (planned from approximate cumulative masses), and a census of the
// bins where the fold steps element by element (binade crossings, ties,
// decisions): their distinct values with multiplicities and smallest ids, in
// list order.  Wave 0 then walks the bins, 64 per step, with a prefix sum of
// their grid sums, up to the first bin that leaves the binade, holds a tie,
// decides, or was planned for another grid; that bin is stepped through its
// distinct values (64 per step the same way, runs of equal values in closed
// form, single exact f32 steps where needed).  A bin the census lacks is
// censused by one more re-read, and the walk resumes where it stopped.
//
// Passes over the row: the maximum, the bin counts and approximate masses,
// the grid sums of total and of the draw (with the census), the grid sums of
// acc once total is known (with a census), and a census round where a walk
// meets a bin the census lacks.
#pragma once

#include "tsm_select.h"

namespace tsm {
namespace nuc {

constexpr uint32_t kNB = kBins;     // value bins
constexpr uint32_t kHS = 2048;      // census capacity: distinct values
constexpr uint32_t kReqMax = 512;   // bins per census
constexpr uint32_t kReqCnt = kHS / 2;      // candidates per census (distinct values at most that many)
constexpr uint32_t kNoBin = 0xFFFFFFFFu;
constexpr uint32_t kNoRun = 0xFFFFFFFFu;
constexpr uint32_t kBL = 4;         // bins per lane in a walk step

// ---- LDS layout (above the re-read pass's penalty table or counts) ----------
constexpr uint32_t kOffE = kOffRank;
constexpr uint32_t kOffECnt = kOffE;                     // u32[kNB] candidates per bin
constexpr uint32_t kOffEMass = kOffECnt + kNB * 4;       // f64[kNB] approximate masses; after planning:
constexpr uint32_t kOffESStart = kOffEMass;              //   f32[kNB] total's fold value at each bin start
constexpr uint32_t kOffEPStart = kOffEMass + kNB * 4;    //   u32[kNB] candidates before each bin
constexpr uint32_t kOffELay = kOffEMass + kNB * 8;       // u32[kNB + 1] weight before each coarse bin, and past the last
constexpr uint32_t kOffEPlan = kOffELay + (kNB + 2) * 4;       // u32[kNB] grid plans
constexpr uint32_t kOffESum = kOffEPlan + kNB * 4;       // u32[4][kNB] grid sums
constexpr uint32_t kOffETie = kOffESum + 4 * kNB * 4;    // u32[4 * kNB / 32] sums with a tie or invalid
constexpr uint32_t kOffETieB = kOffETie + kNB * 4 / 8;   // u32[4 * kNB / 32] sums invalid (or two ties)
constexpr uint32_t kOffEReq = kOffETieB + kNB * 4 / 8;   // u32[kNB / 32] census requests
constexpr uint32_t kOffECpl = kOffEReq + kNB / 8;        // u32[kNB / 32] censused completely
constexpr uint32_t kOffEWpre = kOffECpl + kNB / 8;       // u32[kNB / 32] requests before each word
constexpr uint32_t kOffEBcnt = kOffEWpre + kNB / 8;      // u32[kReqMax] census buckets
constexpr uint32_t kOffEXreq = kOffEBcnt + kReqMax * 4;  // u32[3][kNB / 32] bins each fold expects to step through
constexpr uint32_t kOffETmpB = kOffEXreq + 3 * kNB / 8;  // u32[kNB / 32] request staging
constexpr uint32_t kOffESc = kOffETmpB + kNB / 8;        // u32[32] scalars
constexpr uint32_t kOffEScd = kOffESc + 32 * 4;          // f64[8]
constexpr uint32_t kOffEHKey = kOffEScd + 8 * 8;         // u32[kHS] census keys; runs after census_finish
constexpr uint32_t kOffEHCnt = kOffEHKey + kHS * 4;      // u32[kHS] multiplicities
constexpr uint32_t kOffEHMin = kOffEHCnt + kHS * 4;      // u32[kHS] smallest ids
constexpr uint32_t kOffESort = kOffEHMin + kHS * 4;      // u64[kHS] bucket sort
constexpr uint32_t kOffERunP = kOffESort + kHS * 8;      // f32[kHS] run probabilities
constexpr uint32_t kOffEExp = kOffERunP + kHS * 4;       // u64[32] the expf table
constexpr uint32_t kOffESHi = kOffEExp + 32 * 8;         // f32[kNB] total's value at bin starts, ties up
// crowded coarse bins (see FBins): a count, kCrowd coarse bin ids, then each
// one's cumulative-count table at its kSub + 1 sub-bin edges
constexpr uint32_t kCrowd = 3;
constexpr uint32_t kSub = 256;
constexpr uint32_t kOffECrowd = kOffESHi + kNB * 4;      // u32[4]: slots used, coarse bins
constexpr uint32_t kOffECdf = kOffECrowd + 16;           // u16[kCrowd][kSub + 1] sub-bin edges' CDF (of 65535)
constexpr uint32_t kOffEEnd = kOffECdf + ((kCrowd * (kSub + 1) * 2 + 7) & ~7u);
static_assert(kOffEMass % 8 == 0 && kOffEScd % 8 == 0 && kOffESort % 8 == 0 && kOffEExp % 8 == 0,
              "8-byte LDS records");
static_assert(kOffEEnd <= kOffMisc, "engine LDS overlaps the row's scalars");

__device__ __forceinline__ uint32_t* e_u32(uint32_t off) { return reinterpret_cast<uint32_t*>(lds_base() + off); }
__device__ __forceinline__ uint32_t* e_cnt() { return e_u32(kOffECnt); }
__device__ __forceinline__ double* e_mass() { return reinterpret_cast<double*>(lds_base() + kOffEMass); }
__device__ __forceinline__ float* e_sstart() { return reinterpret_cast<float*>(lds_base() + kOffESStart); }
__device__ __forceinline__ uint32_t* e_pstart() { return e_u32(kOffEPStart); }
__device__ __forceinline__ uint32_t* e_lay() { return e_u32(kOffELay); }
__device__ __forceinline__ uint32_t* e_plan() { return e_u32(kOffEPlan); }
__device__ __forceinline__ uint32_t* e_sum(uint32_t slot) { return e_u32(kOffESum + slot * kNB * 4); }
__device__ __forceinline__ uint32_t* e_tie() { return e_u32(kOffETie); }
__device__ __forceinline__ uint32_t* e_tieb() { return e_u32(kOffETieB); }
__device__ __forceinline__ float* e_shi() { return reinterpret_cast<float*>(lds_base() + kOffESHi); }
__device__ __forceinline__ uint32_t* e_req() { return e_u32(kOffEReq); }
__device__ __forceinline__ uint32_t* e_cpl() { return e_u32(kOffECpl); }
__device__ __forceinline__ uint32_t* e_wpre() { return e_u32(kOffEWpre); }
__device__ __forceinline__ uint32_t* e_bcnt() { return e_u32(kOffEBcnt); }
__device__ __forceinline__ uint32_t* e_xreq(int k) { return e_u32(kOffEXreq + static_cast<uint32_t>(k) * kNB / 8); }
__device__ __forceinline__ uint32_t* e_tmpb() { return e_u32(kOffETmpB); }
__device__ __forceinline__ uint32_t* e_sc() { return e_u32(kOffESc); }
__device__ __forceinline__ double* e_scd() { return reinterpret_cast<double*>(lds_base() + kOffEScd); }
__device__ __forceinline__ uint32_t* e_hkey() { return e_u32(kOffEHKey); }
__device__ __forceinline__ uint32_t* e_hcnt() { return e_u32(kOffEHCnt); }
__device__ __forceinline__ uint32_t* e_hmin() { return e_u32(kOffEHMin); }
__device__ __forceinline__ uint64_t* e_sort() { return reinterpret_cast<uint64_t*>(lds_base() + kOffESort); }
__device__ __forceinline__ float* e_runp() { return reinterpret_cast<float*>(lds_base() + kOffERunP); }
__device__ __forceinline__ uint64_t* e_exptab() { return reinterpret_cast<uint64_t*>(lds_base() + kOffEExp); }
__device__ __forceinline__ uint32_t* e_crowd() { return e_u32(kOffECrowd); }
__device__ __forceinline__ uint16_t* e_cdf(uint32_t slot) {
    return reinterpret_cast<uint16_t*>(lds_base() + kOffECdf) + slot * (kSub + 1u);
}

enum : uint32_t {  // e_sc() words
    SC_FIRST = 0,   // first nonempty bin
    SC_LAST = 1,    // last nonempty bin
    SC_NAN = 2,     // a candidate is NaN
    SC_KLO = 3,     // predicted top-p bins: first, last
    SC_KHI = 4,
    SC_RES = 6,     // walk: result, next bin, position, run, index within run, x bits
    SC_B = 7,
    SC_POS = 8,
    SC_RUN = 9,
    SC_WITHIN = 10,
    SC_X = 11,
    SC_OVF = 12,    // census table full
    SC_CMIN = 13,   // smallest candidate value's total key
    SC_FILED = 15,  // elements filed for the census
};

// Grid plan of a bin, one byte per fold for the lower grid's binade (+128)
// and one of flags.
enum : uint32_t {
    PF_TWO_S = 1u << 24, PF_TWO_R = 1u << 25, PF_TWO_A = 1u << 26,
    PF_MUST_S = 1u << 27, PF_MUST_R = 1u << 28, PF_MUST_A = 1u << 29,
    PF_R = 1u << 30,  // the draw may reach this bin
    PF_REQ = 1u << 31,  // requested of the census (census_clear)
};
enum : int { FK_S = 0, FK_A = 1, FK_R = 2 };  // total (and the kept mass), acc, the draw
enum : uint32_t { SL_S0 = 0, SL_S1 = 1, SL_R0 = 2, SL_R1 = 3 };  // acc reuses slots 0 and 1
enum : uint32_t { W_DONE = 0, W_NEED = 1, W_DECIDED = 2 };

__device__ __forceinline__ uint32_t plan_shift(int k) { return k == FK_S ? 0u : k == FK_R ? 8u : 16u; }
__device__ __forceinline__ uint32_t plan_two(int k) { return k == FK_S ? PF_TWO_S : k == FK_R ? PF_TWO_R : PF_TWO_A; }
__device__ __forceinline__ uint32_t plan_must(int k) {
    return k == FK_S ? PF_MUST_S : k == FK_R ? PF_MUST_R : PF_MUST_A;
}
__device__ __forceinline__ uint32_t slot0(int k) { return k == FK_R ? SL_R0 : SL_S0; }

__device__ __forceinline__ bool tie_bit(uint32_t slot, uint32_t b) {
    const uint32_t i = slot * kNB + b;
    return (e_tie()[i >> 5] >> (i & 31u)) & 1u;
}
// The sum cannot bound the bin's steps (a term too large, a possible wrap, or
// more than one tie).
__device__ __forceinline__ bool bad_bit(uint32_t slot, uint32_t b) {
    const uint32_t i = slot * kNB + b;
    return (e_tieb()[i >> 5] >> (i & 31u)) & 1u;
}
__device__ __forceinline__ bool bit_of(const uint32_t* w, uint32_t b) { return (w[b >> 5] >> (b & 31u)) & 1u; }

// ---- grids -------------------------------------------------------------------
// floor(log2 x) for x > 0 (subnormals: -127, whose grid is that of -126).
__device__ __forceinline__ int binade_of(float x) {
    const int ex = static_cast<int>((__float_as_uint(x) >> 23) & 0xFFu);
    return ex == 0 ? -127 : ex - 127;
}
// log2 of the spacing of floats in binade e.
__device__ __forceinline__ int grid_of(int e) { return (e < -126 ? -126 : e) - 23; }
// The binade whose grid a step from x > 0 rounds on: x's own, or for a
// subtraction from an exact power of two the one below.
__device__ __forceinline__ int step_binade(float x, bool sub) {
    int e = binade_of(x);
    if (sub && (__float_as_uint(x) & 0x7FFFFFu) == 0u && e > -126) e -= 1;
    return e;
}

constexpr uint32_t kTieTerm = 0xFFFFFFFFu;  // tau halfway between grid points
constexpr uint32_t kBigTerm = 0xFFFFFFFEu;  // tau >= 2^(e+1): no grid sum holds its step
// RN_e(tau) in grid units of binade e, or kTieTerm or kBigTerm.
__device__ __forceinline__ uint32_t grid_term(float tau, int e) {
    if (!(tau < ldexpf(1.0f, e + 1))) return kBigTerm;
    const float v = ldexpf(tau, -grid_of(e));  // < 2^24: exact
    const float k = floorf(v);
    const float fr = v - k;
    if (fr == 0.5f) return kTieTerm;
    return static_cast<uint32_t>(k) + (fr > 0.5f ? 1u : 0u);
}

// thr in units of 2^g, rounded up; at most 2^31 (past every fold value's units).
__device__ __forceinline__ uint32_t grid_ceil(float thr, int g) {
    return static_cast<uint32_t>(fminf(ceilf(ldexpf(thr, -g)), 2147483648.0f));
}

__device__ __forceinline__ uint32_t first_lane(uint64_t mask) {
    return mask ? static_cast<uint32_t>(__builtin_ctzll(mask)) : 64u;
}

// ---- bins -----------------------------------------------------------------------
// Fine bins of about equal counts: with C(c) the candidates in coarse bins
// (VBins) before c and n(c) those in c, a value at fraction fr of coarse bin
// c goes to fine bin floor((C(c) + fr * n(c)) * kNB / len).  Monotone in y
// (fine bins keep the list order), equal values share a bin, and a value
// spread that is even inside each coarse bin gives each fine bin about len /
// kNB candidates.  e_lay()[c] = C(c); scale = kNB / len (0: fine = coarse).
//
// A coarse bin whose values are far from even inside it (a dense cluster
// narrower than the bin) can leave one fine bin more candidates than a census
// round takes.  Such a bin (crowded: up to kCrowd of them, cr[]) is laid out
// from a histogram of its own: fr is replaced by the bin's cumulative count
// at fr, interpolated linearly between its kSub sub-bin edges, so its fine
// bins hold about equal counts at the sub-bin's resolution.  The map stays
// monotone in y (the edges' counts never fall) and a function of y alone.
__device__ __forceinline__ float crowd_frac(const uint16_t* F, float fr) {
    const float x = fr * static_cast<float>(kSub);
    const uint32_t j = x < static_cast<float>(kSub - 1u) ? static_cast<uint32_t>(x) : kSub - 1u;
    const float w = x - static_cast<float>(j);  // in [0, 1]
    const float a = static_cast<float>(F[j]), b = static_cast<float>(F[j + 1u]);
    const float v = (a + w * (b - a)) * (1.0f / 65535.0f);
    return v < 1.0f ? v : 1.0f;
}
struct FBins {
    VBins vb;
    float scale;
    uint32_t cr[kCrowd];  // crowded coarse bins laid out from their own sub-histogram (kNoBin: none)
    // (branchless: fmaxf and fminf take a NaN to the other bound)
    __device__ __forceinline__ float frac(float y, uint32_t c) const {
        return fminf(fmaxf(vb.pos(y) - static_cast<float>(c), 0.0f), 1.0f);
    }
    __device__ __forceinline__ uint32_t bin(float y) const {
        const uint32_t c = vb.bin(y);
        if (scale == 0.0f) return c;
        const uint32_t c0 = e_lay()[c], c1 = e_lay()[c + 1u];
        float fr = frac(y, c);
        if (cr[0] != kNoBin) {  // any bin crowded at all (the same for the whole workgroup)
#pragma unroll
            for (uint32_t s = 0; s < kCrowd; s++)
                if (c == cr[s]) fr = crowd_frac(e_cdf(s), fr);
        }
        const float v = (static_cast<float>(c0) + fr * static_cast<float>(c1 - c0)) * scale;
        return min(static_cast<uint32_t>(v), kNB - 1u);
    }
};

// ---- census -------------------------------------------------------------------
// Requested bins in bin order get bucket numbers.
__device__ __forceinline__ uint32_t req_rank(uint32_t b) {
    return e_wpre()[b >> 5] + static_cast<uint32_t>(__popc(e_req()[b >> 5] & ((1u << (b & 31u)) - 1u)));
}

// Empties the census table for the requested bins (at most kReqMax bins and
// kReqCnt candidates, as request_bins leaves them).
__device__ void census_clear() {
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < kHS; i += kBlock) {
        e_hkey()[i] = 0u;
        e_hcnt()[i] = 0u;
        e_hmin()[i] = 0xFFFFFFFFu;
    }
    if (tid < kWave) {  // one request word per lane
        const uint32_t w = e_req()[tid];
        const uint32_t c = static_cast<uint32_t>(__popc(w));
        e_wpre()[tid] = wave_incl_scan(c) - c;
        e_cpl()[tid] = w;
        if (tid == 0) {
            e_sc()[SC_OVF] = 0u;
            e_sc()[SC_FILED] = 0u;
        }
    }
    for (uint32_t b = tid; b < kNB; b += kBlock)
        e_plan()[b] = (e_plan()[b] & ~PF_REQ) | (bit_of(e_req(), b) ? PF_REQ : 0u);
    TSM_LDS_SYNC();
}

__device__ __noinline__ void census_insert(uint32_t key, uint32_t id, uint32_t b) {
    const uint32_t h = (key * 0x9E3779B1u) >> 21;
#pragma unroll 1
    for (uint32_t i = 0; i < 64u; i++) {
        const uint32_t s = (h + i) & (kHS - 1u);
        const uint32_t k = atomicCAS(&e_hkey()[s], 0u, key);
        if (k == 0u || k == key) {
            atomicAdd(&e_hcnt()[s], 1u);
            atomicMin(&e_hmin()[s], id);
            return;
        }
    }
    atomicAnd(&e_cpl()[b >> 5], ~(1u << (b & 31u)));  // no free slot near: the bin stays incomplete
    e_sc()[SC_OVF] = 1u;
}
// A pass files the elements it meets in requested bins as composites (in the
// sort's area, free until census_finish), and the census takes them all at once
// afterwards: one LDS atomic and a store in the pass's loop instead of a
// probe.  What does not fit (one bin requested alone, whatever its count) is
// inserted at once.
__device__ __forceinline__ void census_file(uint32_t key, uint32_t id, uint32_t b) {
    const uint32_t at = atomicAdd(&e_sc()[SC_FILED], 1u);
    if (at < kHS) e_sort()[at] = composite(key, id);
    else census_insert(key, id, b);
}
__device__ __forceinline__ void census_take(const FBins& vb) {
    TSM_LDS_SYNC();
    const uint32_t n = min(e_sc()[SC_FILED], kHS);
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) {
        const uint64_t c = e_sort()[i];
        const uint32_t key = ~static_cast<uint32_t>(c >> 32);
        census_insert(key, static_cast<uint32_t>(c), vb.bin(key_to_float(key)));
    }
}

// Turns the census into runs in list order (value descending): key,
// multiplicity, smallest id and p = exp((y - y0) / t), each bucket (one
// bin) ranked by comparing keys.
__device__ void census_finish(const FBins& vb, float t) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i < kReqMax; i += kBlock) e_bcnt()[i] = 0u;
    TSM_LDS_SYNC();
    for (uint32_t s = tid; s < kHS; s += kBlock) {
        const uint32_t key = e_hkey()[s];
        if (key) atomicAdd(&e_bcnt()[req_rank(vb.bin(key_to_float(key)))], 1u);
    }
    TSM_LDS_SYNC();
    uint32_t total;
    const uint32_t v = tid < kReqMax ? e_bcnt()[tid] : 0u;
    const uint32_t ex = block_excl_scan<kBlock>(v, reinterpret_cast<uint32_t*>(lds_base() + kOffTmp), &total);
    if (tid < kReqMax) e_bcnt()[tid] = ex;
    TSM_LDS_SYNC();
    for (uint32_t s = tid; s < kHS; s += kBlock) {
        const uint32_t key = e_hkey()[s];
        if (key) {
            const uint32_t pos = atomicAdd(&e_bcnt()[req_rank(vb.bin(key_to_float(key)))], 1u);
            e_sort()[pos] = (static_cast<uint64_t>(~key) << 32) | s;
        }
    }
    TSM_LDS_SYNC();
    // e_bcnt()[i] is now the end of bucket i
    constexpr uint32_t kPer = kHS / kBlock;
    uint32_t fin[kPer], fk[kPer], fc[kPer], fm[kPer];
    float fp[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++) {
        const uint32_t pos = tid + k * kBlock;
        fin[k] = 0xFFFFFFFFu;
        if (pos < total) {
            const uint64_t me = e_sort()[pos];
            const uint32_t key = ~static_cast<uint32_t>(me >> 32), slot = static_cast<uint32_t>(me);
            const float y = key_to_float(key);
            const uint32_t ci = req_rank(vb.bin(y));
            const uint32_t bs = ci ? e_bcnt()[ci - 1] : 0u, be = e_bcnt()[ci];
            uint32_t rank = 0;
            for (uint32_t j = bs; j < be; j++) rank += e_sort()[j] < me ? 1u : 0u;
            fin[k] = bs + rank;
            fk[k] = key;
            fc[k] = e_hcnt()[slot];
            fm[k] = e_hmin()[slot];
            fp[k] = glibc_expf_lds((y - vb.vb.y0) / t, e_exptab());
        }
    }
    TSM_LDS_SYNC();
#pragma unroll
    for (uint32_t k = 0; k < kPer; k++)
        if (fin[k] != 0xFFFFFFFFu) {
            e_hkey()[fin[k]] = fk[k];
            e_hcnt()[fin[k]] = fc[k];
            e_hmin()[fin[k]] = fm[k];
            e_runp()[fin[k]] = fp[k];
        }
    TSM_LDS_SYNC();
}

// First run of a censused bin b and the end of its runs: census_finish leaves
// each bucket's runs in its place, and e_bcnt the buckets' ends.
__device__ __forceinline__ void runs_of(uint32_t b, uint32_t* r0, uint32_t* r1) {
    const uint32_t ci = req_rank(b);
    const uint32_t lo = e_bcnt()[ci ? ci - 1u : 0u];
    *r0 = ci ? lo : 0u;
    *r1 = e_bcnt()[ci];
}

// ---- stepping one run of equal terms ----------------------------------------
// m steps of x <- x + tau (S, A) or x <- x - tau (R) in f32, exactly as the
// reference's loop computes them, stopping at the decision (A: x >= thr;
// R: x <= 0).  Steps that stay in one binade without a tie repeat the same
// grid increment and are taken together.  Returns the steps taken (with the
// deciding one).  Wave-uniform scalar code.
template <int K>
__device__ uint32_t run_steps(float& x, float tau, uint32_t m, float thr, bool* decided) {
    constexpr bool sub = K == FK_R;
    uint32_t done = 0;
    *decided = false;
    while (done < m) {
        const float nx = sub ? x - tau : x + tau;
        const bool dec = K == FK_A ? (nx >= thr) : (K == FK_R ? (nx <= 0.0f) : false);
        if (dec) {
            x = nx;
            *decided = true;
            return done + 1;
        }
        if (x > 0.0f) {
            const int e = step_binade(x, sub);
            const int g = grid_of(e);
            const uint32_t c = grid_term(tau, e);
            if (c < kBigTerm) {
                const uint32_t M = static_cast<uint32_t>(ldexpf(x, -g));  // [2^23, 2^24), less for a subnormal x
                const uint32_t left = m - done;
                if (c == 0u) return m;  // every remaining step rounds back to x, and none decides
                uint32_t n;
                if (sub) {
                    n = M > (1u << 23) ? (M - (1u << 23) - 1u) / c : 0u;  // stays above 2^e
                } else {
                    n = ((1u << 24) - M) / c;  // stays at or below 2^(e+1)
                    if (K == FK_A) {
                        const uint32_t mt = grid_ceil(thr, g);
                        const uint32_t nd = mt > M ? (mt - M - 1u) / c : 0u;  // stays below thr
                        n = n < nd ? n : nd;
                    }
                }
                if (n > left) n = left;
                if (n > 0u) {
                    const uint32_t M2 = sub ? M - n * c : M + n * c;  // at most 2^24
                    x = ldexpf(static_cast<float>(M2), g);
                    done += n;
                    continue;
                }
            }
        }
        x = nx;
        done++;
    }
    return done;
}

struct Walk {
    float x;          // the fold's value
    uint32_t b;       // next bin
    uint32_t pos;     // candidates folded so far
    uint32_t run;     // W_DECIDED (in bin b): the deciding run, kNoRun when the census has
                      // been replaced since, and the index within it
    uint32_t within;
};

// The runs [r0, r1) of one bin, in order, folding at most up to candidate
// `lim` (the kept count; ~0 for no limit).  Wave 0.
template <int K>
__device__ uint32_t walk_runs(Walk& w, uint32_t r0, uint32_t r1, float T, float thr, uint32_t lim) {
    constexpr bool sub = K == FK_R;
    const uint32_t lane = lane_id();
    uint32_t i = r0;
    while (i < r1) {
        if (w.x > 0.0f) {
            const int e = step_binade(w.x, sub);
            const int g = grid_of(e);
            const uint32_t M = static_cast<uint32_t>(ldexpf(w.x, -g));
            const uint32_t j = i + lane;
            uint32_t mraw = j < r1 ? e_hcnt()[j] : 0u;
            const uint32_t mpre = wave_incl_scan(mraw) - mraw;
            const uint32_t room = lim - w.pos;  // lim >= w.pos
            uint32_t m = mpre >= room ? 0u : (mraw < room - mpre ? mraw : room - mpre);
            bool ok = j < r1 && m > 0u;
            uint64_t c = 0;
            if (ok) {
                const float p = e_runp()[j];
                const float tau = K == FK_A ? p / T : p;
                const uint32_t t = grid_term(tau, e);
                if (t >= kBigTerm) ok = false;
                else c = static_cast<uint64_t>(m) * t;
            }
            // past 2^25 units a lane leaves the binade anyway: the clamp keeps
            // the prefix sums (and everything below) in 32 bits
            const uint32_t c32 = c > (1ull << 25) ? (1u << 25) : static_cast<uint32_t>(c);
            const uint32_t incl = wave_incl_scan(c32);
            const uint32_t excl = incl - c32;
            bool bad = !ok;
            bool restart = false;
            if (sub) {
                bad |= incl + (1u << 23) >= M;  // the end at or below 2^e
            } else {
                restart = M + excl >= (1u << 24);
                bad |= restart || M + incl > (1u << 24);
                if (K == FK_A) bad |= M + incl >= grid_ceil(thr, g);
            }
            const uint32_t f = first_lane(wave_ballot(bad));
            const uint32_t fl = f < 64u ? f : 63u;
            const uint32_t applied = f < 64u ? wave_read(excl, fl) : wave_read(incl, 63u);
            const uint32_t mapplied = f < 64u ? wave_read(mpre, fl) : wave_read(mpre + m, 63u);
            w.x = ldexpf(static_cast<float>(sub ? M - applied : M + applied), g);
            w.pos += mapplied;
            i += f < 64u ? f : 64u;
            if (f == 64u) continue;
            if (i >= r1 || w.pos >= lim) return W_DONE;
            if (wave_read(restart ? 1u : 0u, fl)) continue;
        }
        // one run exactly
        const uint32_t mraw = e_hcnt()[i];
        const uint32_t room = lim - w.pos;
        const uint32_t m = mraw < room ? mraw : room;
        if (m == 0u) return W_DONE;
        const float p = e_runp()[i];
        const float tau = K == FK_A ? p / T : p;
        bool dec;
        const uint32_t steps = run_steps<K>(w.x, tau, m, thr, &dec);
        w.pos += steps;
        if (dec) {
            w.run = i;
            w.within = steps - 1u;
            return W_DECIDED;
        }
        i++;
    }
    return W_DONE;
}

// The bins from w.b up to bend, in order (wave 0).  A bin is added as its grid
// sum when its plan holds the fold's grid, no step in it ties or runs past
// its sum's range, and the fold stays in its binade and undecided through it;
// otherwise it is stepped through its census runs (W_NEED when the census
// lacks it).  `force` is a bin always stepped through (the kept count's bin,
// whose sums also count candidates past it).  Total's walk records the fold
// value and position at every bin start.
template <int K, int kB = 0>
__device__ uint32_t walk_bins(Walk& w, uint32_t bend, float T, float thr, uint32_t force, uint32_t lim) {
    constexpr bool sub = K == FK_R;
    const uint32_t lane = lane_id();
    while (w.b < bend) {
        bool expand = false;
        if (w.x == 0.0f) {
            // the first step starts from zero: the first nonempty bin is stepped through
            const uint32_t b = w.b + lane;
            const uint32_t n = b < bend ? e_cnt()[b] : 0u;
            const uint32_t f = first_lane(wave_ballot(n > 0u || b >= bend));
            if (K == FK_S && b < bend && lane <= f) {
                if (kB != 2) e_sstart()[b] = 0.0f;
                if (kB != 1) e_shi()[b] = 0.0f;
                if (kB != 2) e_pstart()[b] = w.pos;  // the ties-up walk runs beside the ties-down one
            }
            if (f == 64u) {
                w.b += 64u;
                continue;
            }
            w.b += f;
            if (w.b >= bend) break;
            expand = true;
        } else {
            // kBL bins per lane: lane l takes bins w.b + kBL*l .. + kBL-1
            const int e = step_binade(w.x, sub);
            const int g = grid_of(e);
            const uint32_t M = static_cast<uint32_t>(ldexpf(w.x, -g));
            const uint32_t mthr = K == FK_A ? grid_ceil(thr, g) : 0u;
            const uint32_t bl = w.b + kBL * lane;
            uint32_t nj[kBL], cj[kBL];
            bool okj[kBL];
            uint32_t ln = 0, lc = 0;
            // every word of the lane's bins first, whatever the plans turn out
            // to say: one wait for LDS instead of one a bin and condition (with
            // the runs found by their bucket: 60 -> 40 us for total's two walks
            // of a row, 80 -> 60 us for the draw's)
            uint32_t pj[kBL], s0[kBL], s1[kBL], t0[kBL], t1[kBL], a0[kBL], a1[kBL];
#pragma unroll
            for (uint32_t j = 0; j < kBL; j++) {
                const uint32_t b = min(bl + j, kNB - 1u), i0 = slot0(K) * kNB + b, i1 = i0 + kNB;
                nj[j] = e_cnt()[b];
                pj[j] = e_plan()[b];
                s0[j] = e_sum(slot0(K))[b];
                s1[j] = e_sum(slot0(K) + 1u)[b];
                t0[j] = e_tie()[i0 >> 5] >> (i0 & 31u);
                t1[j] = e_tie()[i1 >> 5] >> (i1 & 31u);
                a0[j] = e_tieb()[i0 >> 5] >> (i0 & 31u);
                a1[j] = e_tieb()[i1 >> 5] >> (i1 & 31u);
            }
#pragma unroll
            for (uint32_t j = 0; j < kBL; j++) {
                const uint32_t b = bl + j;
                const uint32_t n = b < bend ? nj[j] : 0u, pw = pj[j];
                // the bin's sum for the fold's grid, if it has one
                const int g0 = static_cast<int>((pw >> plan_shift(K)) & 0xFFu) - 128;
                const bool planned = !(pw & plan_must(K)) && (K != FK_R || (pw & PF_R));
                const bool low = planned && e == g0, high = planned && e == g0 + 1 && (pw & plan_two(K));
                const bool tie = ((high ? t1[j] : t0[j]) & 1u) != 0u, bad = ((high ? a1[j] : a0[j]) & 1u) != 0u;
                // exact walks step through a bin with a tie; bound walks take its
                // lower (kB 1) or upper (kB 2) end
                bool ok = (low || high) && b != force && (kB == 0 ? !tie : !bad);
                uint32_t c = min(high ? s1[j] : s0[j], 1u << 25) + (kB == 2 && tie ? 1u : 0u);
                const bool take = ok && n != 0u;
                c = take ? c : 0u;
                ok = b < bend && (ok || n == 0u);  // past bend: the end marker; an empty bin passes
                // past 2^25 units a bin leaves the binade anyway: the clamps keep
                // the prefix sums in 32 bits
                cj[j] = min(c, 1u << 25);
                nj[j] = n;
                okj[j] = ok;
                ln += n;
                lc = min(lc + cj[j], 1u << 25);
            }
            const uint32_t npre = wave_incl_scan(ln) - ln;
            const uint32_t cpre = wave_incl_scan(lc) - lc;
            uint32_t jb = kBL;  // the lane's first bin the sums cannot take
            bool restart = false;
            uint32_t pre = cpre;  // at most 64 * 2^25, and four bins more: 32 bits
            uint32_t np = npre;
            uint32_t pre_at = 0;
            uint32_t np_at = 0;
#pragma unroll
            for (uint32_t j = 0; j < kBL; j++) {
                const uint32_t start = sub ? M - pre : M + pre;
                bool bad = !okj[j];
                bool rs = false;
                if (sub) {
                    bad |= nj[j] > 0u && pre + cj[j] + (1u << 23) >= M;  // the end at or below 2^e
                } else {
                    const uint32_t end = start + cj[j];
                    rs = start >= (1u << 24);
                    bad |= rs || end > (1u << 24);
                    if (K == FK_A) bad |= nj[j] > 0u && end >= mthr;
                }
                if (jb == kBL) {
                    if (K == FK_S && bl + j < bend) {
                        const float sv = ldexpf(static_cast<float>(start), g);
                        if (kB != 2) e_sstart()[bl + j] = sv;
                        if (kB != 1) e_shi()[bl + j] = sv;
                        if (kB != 2) e_pstart()[bl + j] = w.pos + np;
                    }
                    if (bad) {
                        jb = j;
                        restart = rs;
                        pre_at = pre;
                        np_at = np;
                    }
                }
                pre += cj[j];
                np += nj[j];
            }
            const uint32_t f = first_lane(wave_ballot(jb < kBL));
            // lanes after f recorded bin starts past the stop; the next step
            // writes them again from the right value
            if (f == 64u) {
                const uint32_t applied = wave_read(pre, 63u);  // cpre + lc of the last lane
                w.x = ldexpf(static_cast<float>(sub ? M - applied : M + applied), g);
                w.pos += wave_read(np, 63u);
                w.b += kBL * 64u;
                continue;
            }
            const uint32_t applied = wave_read(pre_at, f);
            w.x = ldexpf(static_cast<float>(sub ? M - applied : M + applied), g);
            w.pos += wave_read(np_at, f);
            w.b = wave_read(bl + jb, f);
            if (w.b >= bend) break;
            if (wave_read(restart ? 1u : 0u, f)) continue;
            expand = true;
        }
        if (expand) {
            const uint32_t bb = w.b;
            if (!bit_of(e_cpl(), bb)) return W_NEED;
            uint32_t r0, r1;
            runs_of(bb, &r0, &r1);
            const uint32_t res = walk_runs<K>(w, r0, r1, T, thr, lim);
            if (res == W_DECIDED) return res;
            w.b = bb + 1u;
        }
    }
    return W_DONE;
}

__device__ __forceinline__ void set_bit(uint32_t* w, uint32_t b) { atomicOr(&w[b >> 5], 1u << (b & 31u)); }

// Does fold K expect to step through bin b (a predicted crossing or decision,
// a bin planned without a grid, or a step its sums could not take; for the
// exact walk also a tie, which the bound walks take as two ends)?
__device__ __forceinline__ bool fold_needs(int k, uint32_t b, bool exact) {
    const uint32_t pw = e_plan()[b];
    if (bit_of(e_xreq(k), b) || (pw & plan_must(k))) return true;
    if (k == FK_R && !(pw & PF_R)) return false;
    const uint32_t s0 = slot0(k);
    return exact ? (tie_bit(s0, b) || tie_bit(s0 + 1u, b)) : (bad_bit(s0, b) || bad_bit(s0 + 1u, b));
}

// ---- passes ----------------------------------------------------------------
// tau's grid units for the sums of slot `slot` (the grid of binade g, g >=
// -126); a step that cannot be summed, or a sum that could pass 2^32 over the
// bin's n candidates, marks the bin's sum invalid.  The same units as
// grid_term, by rounding tau / grid to the nearest integer: a tie is where that
// moved it by a half.
__device__ __forceinline__ void add_term(uint32_t slot, uint32_t b, float tau, int g, uint32_t n) {
    const float v = ldexpf(tau, 23 - g);
    const float r = rintf(v), d = v - r;
    const bool tie = fabsf(d) == 0.5f;
    // a tie takes its lower end; the tie bit says it may be one more
    const uint32_t t = static_cast<uint32_t>(tie ? floorf(v) : r);
    const bool bad = !(v < 16777216.0f) || (n > 255u && static_cast<uint64_t>(t) * n >= (1ull << 32));
    atomicAdd(&e_sum(slot)[b], bad ? 0u : t);
    if (bad || tie) {
        const uint32_t i = slot * kNB + b;
        const uint32_t bit = 1u << (i & 31u);
        const uint32_t old = atomicOr(&e_tie()[i >> 5], bit);
        if (bad || (old & bit)) atomicOr(&e_tieb()[i >> 5], bit);
    }
}

// a / b rounded to f32, for f32 a and b with inv = 1 / b in f64: the product's
// relative error is below 2^-51, and no quotient of two f32 values lies within
// 2^-49 of the middle between two f32 values (its distance from one is a
// nonzero multiple of 2^-24 / b in units of the middle's last place), so it
// rounds as the quotient does.  A subnormal quotient may round otherwise, which
// shows nowhere: exp of (y - y0) / t is 1 then, and a p / total that small is
// none of acc's grid units, whose first term is 1 / total.  A third of the
// instructions of the f32 division.
__device__ __forceinline__ float quotient(float a, double inv) {
    return static_cast<float>(static_cast<double>(a) * inv);
}

enum : int { EP_HIST = 0, EP_SR = 1, EP_A = 2, EP_CENSUS = 3, EP_SUB = 4 };

// One re-read of the row for the engine, its candidates (filter q, in total
// order) handled by mode:
//   EP_HIST    candidates and approximate masses (hardware exp2) per bin, the
//              smallest candidate's key, whether a candidate is NaN;
//   EP_SR      the grid sums of total and the draw, and the census;
//   EP_A       the grid sums of acc (terms p / T), and the census;
//   EP_CENSUS  the census alone;
//   EP_SUB     the crowded coarse bins' sub-histograms (kSub bins each, in
//              e_hkey, which holds no census yet).
// The row is read by row_blocks, four elements at a time.
template <int kMode>
__device__ __noinline__ void eng_pass(Fin& f_in, const Filt& q_in, const FBins& vb_in, float T) {
    const Fin f = f_in;  // a private copy: its fields stay in registers across LDS atomics
    // the same for every lane: in scalar registers
    Filt q = q_in;
    q.use_cut = wave_uniform(q.use_cut ? 1u : 0u) != 0u;
    q.use_max = wave_uniform(q.use_max ? 1u : 0u) != 0u;
    q.need_allowed = wave_uniform(q.need_allowed ? 1u : 0u) != 0u;
    q.use_minp = wave_uniform(q.use_minp ? 1u : 0u) != 0u;
    FBins vb = vb_in;
    vb.vb.y0 = wave_uniform_f(vb.vb.y0);
    vb.vb.mul = wave_uniform_f(vb.vb.mul);
    vb.scale = wave_uniform_f(vb.scale);
#pragma unroll
    for (uint32_t s = 0; s < kCrowd; s++) vb.cr[s] = wave_uniform(vb.cr[s]);
    const uint32_t tid = threadIdx.x;
    if (kMode == EP_HIST) {
        for (uint32_t i = tid; i < kNB; i += kBlock) {
            e_cnt()[i] = 0u;
            e_mass()[i] = 0.0;
        }
        if (tid == 0) {
            e_sc()[SC_NAN] = 0u;
            e_sc()[SC_CMIN] = 0xFFFFFFFFu;
        }
    } else if (kMode == EP_SUB) {
        for (uint32_t i = tid; i < kCrowd * kSub; i += kBlock) e_hkey()[i] = 0u;
    } else if (kMode == EP_SR || kMode == EP_A) {
        const uint32_t nslot = kMode == EP_SR ? 4u : 2u;
        for (uint32_t i = tid; i < nslot * kNB; i += kBlock) e_sum(0)[i] = 0u;
        for (uint32_t i = tid; i < nslot * kNB / 32u; i += kBlock) {
            e_tie()[i] = 0u;
            e_tieb()[i] = 0u;
        }
    }
    TSM_LDS_SYNC();
    const float t = wave_uniform_f(f.m.t);
    const float y0 = vb.vb.y0;
    const float l2t = 1.4426950408889634f / t;
    const double invt = 1.0 / static_cast<double>(t), invT = 1.0 / static_cast<double>(T);
    const uint64_t* tab = e_exptab();
    float ymin = INFINITY;
    bool nan = false;
    const TSM_GLOBAL_AS uint32_t* mrow = global_as(wave_uniform_p(f.mrow));
    // without a cut every id is a candidate, NaNs too: they fail a compare with
    // the cut, as they should with one, and are taken up by `more`
    const bool nocut = !q.use_cut, more = nocut || q.use_max || q.need_allowed || q.use_minp;
    const float cut = nocut ? -INFINITY : wave_uniform_f(q.cut);

    row_blocks(f, [&](uint32_t id0, uint32_t in, const float (&)[4], const float (&y)[4]) __attribute__((always_inline)) {
        bool keep[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) keep[e] = ((in >> e) & 1u) && y[e] >= cut;
        if (more) {
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                const uint32_t id = id0 + e;
                bool k = keep[e] || (nocut && ((in >> e) & 1u));
                if (q.use_max) k = k && composite(total_key(y[e]), id) <= q.max_comp;
                if (q.need_allowed && k) k = (mrow[id >> 5] >> (id & 31u)) & 1u;
                if (q.use_minp && k) {
                    k = !(y[e] < q.minp_lo);
                    if (k && !(y[e] >= q.minp_hi))
                        k = glibc_expf_lds(quotient(y[e] - q.y0, invt), tab) >= q.minp;
                }
                keep[e] = k;
            }
        }
        if (kMode == EP_SUB) {
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                if (!(keep[e] && y[e] == y[e])) continue;
                const uint32_t c = vb.vb.bin(y[e]);
#pragma unroll
                for (uint32_t s = 0; s < kCrowd; s++) {
                    if (c != vb.cr[s]) continue;
                    const float x = vb.frac(y[e], c) * static_cast<float>(kSub);
                    const uint32_t j = x < static_cast<float>(kSub - 1u) ? static_cast<uint32_t>(x) : kSub - 1u;
                    atomicAdd(&e_hkey()[s * kSub + j], 1u);
                }
            }
            return;
        }
        // the four elements' lookups first, then their updates: the LDS reads
        // of one element do not wait behind another's atomics
        uint32_t b[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) b[e] = vb.bin(y[e]);
        if (kMode == EP_HIST) {
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                const bool isnan = y[e] != y[e];
                nan |= keep[e] && isnan;
                if (keep[e] && !isnan) {
                    const double m = static_cast<double>(__builtin_amdgcn_exp2f((y[e] - y0) * l2t));
                    ymin = fminf(ymin, y[e]);
                    atomicAdd(&e_cnt()[b[e]], 1u);
                    atomicAdd(&e_mass()[b[e]], m);
                }
            }
            return;
        }
        uint32_t pw[4], nb[4];
        float p[4];
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++) {
            pw[e] = e_plan()[b[e]];
            if (kMode != EP_CENSUS) {
                nb[e] = e_cnt()[b[e]];
                p[e] = glibc_expf_lds(quotient(y[e] - y0, invt), tab);
                if (kMode == EP_A) p[e] = quotient(p[e], invT);
            }
        }
        if (kMode == EP_SR || kMode == EP_A) {
            constexpr uint32_t sh = kMode == EP_SR ? 0u : 16u;
            constexpr uint32_t must = kMode == EP_SR ? PF_MUST_S : PF_MUST_A, two = kMode == EP_SR ? PF_TWO_S : PF_TWO_A;
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                const int g = static_cast<int>((pw[e] >> sh) & 0xFFu) - 128;
                if (keep[e] && !(pw[e] & must)) {
                    add_term(SL_S0, b[e], p[e], g, nb[e]);
                    if (pw[e] & two) add_term(SL_S1, b[e], p[e], g + 1, nb[e]);
                }
            }
        }
        if (kMode == EP_SR) {
#pragma unroll
            for (uint32_t e = 0; e < 4u; e++) {
                const int g = static_cast<int>((pw[e] >> 8) & 0xFFu) - 128;
                if (keep[e] && (pw[e] & PF_R) && !(pw[e] & PF_MUST_R)) {
                    add_term(SL_R0, b[e], p[e], g, nb[e]);
                    if (pw[e] & PF_TWO_R) add_term(SL_R1, b[e], p[e], g + 1, nb[e]);
                }
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < 4u; e++)
            if (keep[e] && (pw[e] & PF_REQ)) census_file(total_key(y[e]), id0 + e, b[e]);
    });
    if (kMode == EP_SR || kMode == EP_A || kMode == EP_CENSUS) census_take(vb);
    if (kMode == EP_HIST) {
        TSM_LDS_SYNC();
        const uint32_t kmin = wave_min(ymin == INFINITY ? 0xFFFFFFFFu : total_key(ymin));
        if (lane_id() == 0 && kmin != 0xFFFFFFFFu) atomicMin(&e_sc()[SC_CMIN], kmin);
        if (nan) e_sc()[SC_NAN] = 1u;
    }
    TSM_LDS_SYNC();
}

// ---- plans ---------------------------------------------------------------------
// Relative error allowed between a fold and the approximate cumulative masses
// it is planned from (hardware exp2 terms, f64 sums; the f32 fold's own
// rounding drift): a bin whose fold value may lie on either side of a power of
// two gets both grids, or no sum at all when the range spans more.
constexpr double kPlanEps = 1e-4;
// The same for predicting where a fold will step value by value (census
// requests): tighter, since a miss costs a census round, not a wrong result.
constexpr double kPredEps = 2e-5;
// ... and, of the total, for the draw's value.
constexpr double kDrawSlack = 1e-5;

__device__ __forceinline__ void plan_range(double lo, double hi, bool sub, uint32_t shift, uint32_t two,
                                           uint32_t must, uint32_t* pw) {
    const int e_lo = step_binade(static_cast<float>(lo), sub);
    const int e_hi = binade_of(static_cast<float>(hi));
    if (!(lo > 0.0) || e_hi - e_lo >= 2 || e_lo < -126) {
        *pw |= must;
        return;
    }
    *pw |= static_cast<uint32_t>(e_lo + 128) << shift;
    if (e_hi > e_lo) *pw |= two;
}

// What a fold moves by over a bin of n candidates of approximate mass m when
// its value there is about x: each step rounds to the grid of x's binade, which
// drops or doubles terms not far above the grid (f32 folds of 150,000 terms end
// up to 2e-4 off the sum because of it).  A bin is narrow: its terms are taken
// as spread evenly over a stretch `wide` of their mean wide, which holds at most
// one step of the rounding.
__device__ __forceinline__ double fold_mass(double m, uint32_t n, double x, bool sub, double wide) {
    if (!n || !(x > 0.0)) return m;
    const double unit = ldexp(1.0, grid_of(step_binade(static_cast<float>(x), sub)));
    const double v = m / (static_cast<double>(n) * unit);
    if (!(v < 64.0)) return m;
    const double k = floor(v), up = (v * (1.0 + 0.5 * wide) - (k + 0.5)) / (v * wide);
    return static_cast<double>(n) * (k + fmin(fmax(up, 0.0), 1.0)) * unit;
}
// This thread's two bins' masses and the cumulative ones before them, as total's
// fold and as the draw's (from r = u * kept) see them.
struct FoldView {
    double S[2], ms[2], R[2], mr[2];  // cumulative, own
    double tot, kept;                 // total's fold; about its part up to top_p
};
// `wide`: a coarse bin's width, relative to its terms.
__device__ FoldView fold_view(Fin& f, const double (&m)[2], const uint32_t (&c)[2], float u, bool draw, bool topp,
                              double wide) {
    FoldView w;
    double t0;
    const double P0 = block_excl_scan_f64(m[0] + m[1], f.miscd() + 8, &t0);
    w.ms[0] = fold_mass(m[0], c[0], P0, false, wide);
    w.ms[1] = fold_mass(m[1], c[1], P0 + m[0], false, wide);
    w.S[0] = block_excl_scan_f64(w.ms[0] + w.ms[1], f.miscd() + 8, &w.tot);
    w.S[1] = w.S[0] + w.ms[0];
    w.kept = topp ? fmin(static_cast<double>(f.P.top_p), 1.0) * w.tot : w.tot;
    const double r0 = static_cast<double>(u) * w.kept;
    w.mr[0] = draw ? fold_mass(m[0], c[0], r0 - w.S[0], true, wide) : w.ms[0];
    w.mr[1] = draw ? fold_mass(m[1], c[1], r0 - w.S[1], true, wide) : w.ms[1];
    double rt = 0.0;
    w.R[0] = draw ? block_excl_scan_f64(w.mr[0] + w.mr[1], f.miscd() + 8, &rt) : w.S[0];
    w.R[1] = w.R[0] + w.mr[0];
    return w;
}

// Plans of total and the draw from the approximate masses, with the bins each
// is expected to step through.  Two bins per thread.
__device__ void plan_sr(Fin& f, float u, bool draw, bool topp, double wide) {
    const uint32_t tid = threadIdx.x;
    const uint32_t b0 = 2 * tid;
    for (uint32_t i = tid; i < 3u * kNB / 32u; i += kBlock) e_xreq(0)[i] = 0u;
    if (tid == 0) {
        e_sc()[SC_KLO] = 0xFFFFFFFFu;
        e_sc()[SC_KHI] = 0u;
    }
    const double mb[2] = {e_mass()[b0], e_mass()[b0 + 1]};
    const uint32_t cb[2] = {e_cnt()[b0], e_cnt()[b0 + 1]};
    const FoldView w = fold_view(f, mb, cb, u, draw, topp, wide);  // barriers order the clears above
    const double tot = w.tot;
    const double tp = static_cast<double>(f.P.top_p);
    const double eps2 = kPredEps;
    if (topp) {
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (cb[k] && (w.S[k] + w.ms[k]) / tot >= tp - eps2 && w.S[k] / tot <= tp + eps2) {
                atomicMin(&e_sc()[SC_KLO], b0 + k);
                atomicMax(&e_sc()[SC_KHI], b0 + k);
            }
    }
    TSM_LDS_SYNC();
    const uint32_t klo = e_sc()[SC_KLO], khi = e_sc()[SC_KHI];
#pragma unroll
    for (int k = 0; k < 2; k++) {  // the kept mass's bounds: cumulative masses at the region's ends
        if (topp && klo != 0xFFFFFFFFu && b0 + k == klo) e_scd()[0] = w.S[k];
        if (topp && klo != 0xFFFFFFFFu && b0 + k == khi) e_scd()[1] = w.S[k] + w.ms[k];
    }
    TSM_LDS_SYNC();
    double M_lo = tot, M_hi = tot;
    if (topp && klo != 0xFFFFFFFFu) {
        M_lo = e_scd()[0];
        M_hi = e_scd()[1];
    }
    M_lo *= 1.0 - kPredEps;
    M_hi *= 1.0 + kPredEps;
    const double du = static_cast<double>(u);
    // r carries what the estimates leave of the drift of both f32 folds over
    // the whole row: an absolute margin.  A draw that ends deep in the tail
    // stays inside the margin for long, and every bin there is stepped value by
    // value.
    const double slack = kDrawSlack * tot;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const uint32_t b = b0 + k;
        if (!cb[k]) {
            e_plan()[b] = PF_MUST_S | PF_MUST_R | PF_MUST_A;
            continue;
        }
        uint32_t pw = 0;
        // total: the fold value at the bin's start is about S
        const double slo = w.S[k] * (1.0 - kPlanEps), shi = w.S[k] * (1.0 + kPlanEps);
        plan_range(slo, shi, false, 0u, PF_TWO_S, PF_MUST_S, &pw);
        if ((pw & PF_MUST_S) || binade_of(static_cast<float>((w.S[k] + w.ms[k]) * (1.0 + kPlanEps))) !=
                                     binade_of(static_cast<float>(slo)))
            set_bit(e_xreq(FK_S), b);
        if (draw) {
            // the draw: r at the bin's start is about u * M - R
            const double rlo = du * M_lo - w.R[k] * (1.0 + kPredEps) - slack,
                         rhi = du * M_hi - w.R[k] * (1.0 - kPredEps) + slack;
            if (rhi > 0.0) {
                pw |= PF_R;
                plan_range(rlo, rhi, true, 8u, PF_TWO_R, PF_MUST_R, &pw);
                // r may leave its binade (or reach zero) in this bin when the
                // lowest end value and the highest start value lie in
                // different binades
                const double elo = rlo - w.mr[k] * (1.0 + kPredEps);
                if ((pw & PF_MUST_R) || !(elo > 0.0) ||
                    binade_of(static_cast<float>(elo)) != step_binade(static_cast<float>(rhi), true))
                    set_bit(e_xreq(FK_R), b);
            }
        }
        if (topp && klo != 0xFFFFFFFFu && b >= klo && b <= khi) {
            set_bit(e_xreq(FK_A), b);
            if (draw) set_bit(e_xreq(FK_R), b);
        }
        e_plan()[b] = pw;
    }
    TSM_LDS_SYNC();
}

// acc's plan once total's walk has left the fold value at every bin start.
__device__ void plan_a(float T, float top_p) {
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b < kNB; b += kBlock) {
        const uint32_t n = e_cnt()[b];
        if (!n) continue;
        uint32_t pw = e_plan()[b] & ~(0xFFu << 16 | PF_TWO_A | PF_MUST_A);
        const double s = static_cast<double>(e_sstart()[b]);
        const double s_end = b + 1 < kNB ? static_cast<double>(e_sstart()[b + 1]) : static_cast<double>(T);
        const double a = s / T, a_end = s_end / T;
        const double lo = a * (1.0 - kPlanEps), hi = a * (1.0 + kPlanEps);
        plan_range(lo, hi, false, 16u, PF_TWO_A, PF_MUST_A, &pw);
        const bool before = a <= top_p * (1.0 + kPredEps);  // acc stops at top_p
        const bool decides = before && a_end * (1.0 + kPredEps) >= top_p;
        if (before && ((pw & PF_MUST_A) || decides ||
                       binade_of(static_cast<float>(a_end * (1.0 + kPredEps))) !=
                           binade_of(static_cast<float>(a * (1.0 - kPredEps)))))
            set_bit(e_xreq(FK_A), b);
        e_plan()[b] = pw;
    }
    TSM_LDS_SYNC();
}

// Clears the tie bits of slots 0 and 1 (total's, before acc's sums).
__device__ __forceinline__ void clear_ties01() {
    for (uint32_t i = threadIdx.x; i < 2u * kNB / 32u; i += kBlock) {
        e_tie()[i] = 0u;
        e_tieb()[i] = 0u;
    }
    TSM_LDS_SYNC();
}

// Keeps the lowest bins of the bitmap w (one word per lane of wave 0) while
// their candidates stay within cap_cnt and their number within cap_bins (the
// lowest bin is kept whatever its count when `first` is set); returns the
// candidates and bins kept, summed over the wave.
__device__ uint2 trim_bins(uint32_t& w, uint32_t cap_cnt, uint32_t cap_bins, bool first) {
    const uint32_t lane = lane_id();
    uint32_t cnt = 0;
    for (uint32_t bits = w; bits; bits &= bits - 1u) cnt += e_cnt()[32u * lane + static_cast<uint32_t>(__builtin_ctz(bits))];
    const uint32_t nb = static_cast<uint32_t>(__popc(w));
    const uint32_t pc = wave_incl_scan(cnt) - cnt, pb = wave_incl_scan(nb) - nb;
    const uint32_t anyb = first ? first_lane(wave_ballot(w != 0u)) : 64u;  // lane holding the lowest bin
    if (pc + cnt > cap_cnt || pb + nb > cap_bins) {
        uint32_t kept = 0, c = pc, k = pb;
        for (uint32_t bits = w; bits; bits &= bits - 1u) {
            const uint32_t i = static_cast<uint32_t>(__builtin_ctz(bits));
            const uint32_t ci = e_cnt()[32u * lane + i];
            const bool must = lane == anyb && kept == 0u && pc == 0u && pb == 0u;
            if (!must && (c + ci > cap_cnt || k + 1u > cap_bins)) break;
            kept |= 1u << i;
            c += ci;
            k++;
        }
        w = kept;
    }
    uint32_t kc = 0;
    for (uint32_t bits = w; bits; bits &= bits - 1u) kc += e_cnt()[32u * lane + static_cast<uint32_t>(__builtin_ctz(bits))];
    return make_uint2(wave_sum(kc), wave_sum(static_cast<uint32_t>(__popc(w))));
}

// Requests of a census round for fold K stopped at bin `from`: that bin and
// the bins after it that fold K expects to step through, then, in the room
// left, those of the folds still to come (acc's when acc_next, the draw's
// when draw).  Within kReqCnt candidates and kReqMax bins, lowest bins first.
__device__ void request_round(int K, uint32_t from, bool draw, bool acc_next, bool exact, bool whole = false) {
    // every thread judges its bins, a wave's 64 by ballots; wave 0 then trims
    // the two bitmaps, a word a lane (e_req: this fold's, e_tmpb: the others')
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b < kNB; b += kBlock) {
        bool now = false, after = false;
        if (e_cnt()[b]) {
            const bool needs = fold_needs(K, b, exact);
            now = b == from || (b > from && needs);
            after = !now && ((whole && needs) ||
                             (K == FK_S && ((acc_next && bit_of(e_xreq(FK_A), b)) || (draw && fold_needs(FK_R, b, false)))) ||
                             (K == FK_A && draw && fold_needs(FK_R, b, false)));
        }
        const uint64_t bn = wave_ballot(now), ba = wave_ballot(after);
        if (lane_id() < 2u) {
            const uint32_t w = (b & ~(kWave - 1u)) / 32u + lane_id();
            e_req()[w] = static_cast<uint32_t>(lane_id() ? bn >> 32 : bn);
            e_tmpb()[w] = static_cast<uint32_t>(lane_id() ? ba >> 32 : ba);
        }
    }
    TSM_LDS_SYNC();
    if (tid < kWave) {
        uint32_t cur = e_req()[tid], later = e_tmpb()[tid];
        const uint2 used = trim_bins(cur, kReqCnt, kReqMax, true);
        const uint32_t room_c = used.x < kReqCnt ? kReqCnt - used.x : 0u;
        const uint32_t room_b = used.y < kReqMax ? kReqMax - used.y : 0u;
        trim_bins(later, room_c, room_b, false);
        e_req()[tid] = cur | later;
    }
    TSM_LDS_SYNC();
}

// The draw's expectations past bin `from`, where its walks stand at r in
// [xlo, xhi], from what the bins' sums on the planned grids (else total's fold)
// say they take: a bin whose plan lacks the grid r will be on, or in which r
// leaves its binade, is one to step through; the others, and those from bend
// on, are not.  The plan's own estimate can be off by more than its margin
// where the candidates of a bin share one value (logits rounded to bf16), and
// every bin up to a crossing's real place then asked for a pass over the row of
// its own.  256 rows of 151,936 such ids at sigma 2, draws near 1: 7.9 -> 2.0
// ms; with top_p 0.98 10.8 -> 1.9 ms, at most 4 census rounds a row for 117.
__device__ __noinline__ void replan_draw(float xlo, float xhi, uint32_t from, uint32_t bend) {
    const uint32_t b0 = 2u * threadIdx.x;
    double m[2], all;
#pragma unroll
    for (uint32_t k = 0; k < 2u; k++) {
        const uint32_t b = b0 + k, pw = e_plan()[b];
        m[k] = 0.0;
        if (b < from || b >= bend || !e_cnt()[b]) continue;
        if ((pw & PF_R) && !(pw & PF_MUST_R) && !bad_bit(SL_R0, b))
            m[k] = ldexp(static_cast<double>(e_sum(SL_R0)[b]), grid_of(static_cast<int>((pw >> 8) & 0xFFu) - 128));
        else if (b + 1u < kNB)
            m[k] = fmax(static_cast<double>(e_sstart()[b + 1u]) - static_cast<double>(e_sstart()[b]), 0.0);
    }
    double P = block_excl_scan_f64(m[0] + m[1], reinterpret_cast<double*>(lds_base() + kOffMiscD) + 8, &all);
    uint32_t pair = 0;
#pragma unroll
    for (uint32_t k = 0; k < 2u; k++) {
        const uint32_t b = b0 + k, pw = e_plan()[b];
        const double eps = 1e-5 * P + 1e-6 * xhi, hi = xhi - P + eps, lo = xlo - P - m[k] - eps;
        P += m[k];
        bool need = b < bend && e_cnt()[b] && hi > 0.0;
        if (need && lo > 0.0) {
            const int e = step_binade(static_cast<float>(hi), true), g0 = static_cast<int>((pw >> 8) & 0xFFu) - 128;
            const bool held = (pw & PF_R) && !(pw & PF_MUST_R) && (e == g0 || (e == g0 + 1 && (pw & PF_TWO_R)));
            need = !held || step_binade(static_cast<float>(lo), true) != e;
        }
        pair |= need ? 1u << k : 0u;
    }
    // a word of the bitmap per 16 lanes; the bins up to `from` keep theirs
    uint32_t word = pair << (b0 & 31u);
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) word |= __shfl_xor(word, o, kWave);
    if ((b0 & 31u) == 0u) {
        const uint32_t keep = from >= b0 + 31u ? ~0u : from < b0 ? 0u : (2u << (from - b0)) - 1u;
        uint32_t* w = &e_xreq(FK_R)[b0 >> 5];
        *w = (*w & keep) | (word & ~keep);
    }
    TSM_LDS_SYNC();
}

// Fold K's walk on wave 0 from w, with census rounds wherever the census
// lacks a bin the walk must step through.  Returns W_DONE or W_DECIDED with w
// updated, or W_NEED when a bin holds more distinct values than the census.
template <int K, int kB = 0>
__device__ __noinline__ uint32_t run_walk(Fin& f_in, const Filt& q_in, const FBins& vb_in, Walk& w_io,
                                          uint32_t bend, float T, float thr, uint32_t force, uint32_t lim,
                                          bool draw, bool acc_next) {
    Fin f = f_in;  // a private copy: its fields stay in registers across LDS atomics
    const Filt q = q_in;
    const FBins vb = vb_in;
    const uint32_t tid = threadIdx.x;
    Walk w = w_io;
    uint32_t last_from = kNoBin;
    bool alone = false;
    for (;;) {
        if (tid < kWave) {
            const uint32_t res = walk_bins<K, kB>(w, bend, T, thr, force, lim);
            if (tid == 0) {
                e_sc()[SC_RES] = res;
                e_sc()[SC_B] = w.b;
                e_sc()[SC_POS] = w.pos;
                e_sc()[SC_RUN] = w.run;
                e_sc()[SC_WITHIN] = w.within;
                e_sc()[SC_X] = __float_as_uint(w.x);
            }
        }
        TSM_LDS_SYNC();
        const uint32_t res = e_sc()[SC_RES];
        w.b = e_sc()[SC_B];
        w.pos = e_sc()[SC_POS];
        w.run = e_sc()[SC_RUN];
        w.within = e_sc()[SC_WITHIN];
        w.x = __uint_as_float(e_sc()[SC_X]);
        TSM_LDS_SYNC();
        if (res != W_NEED) {
            w_io = w;
            return res;
        }
        if (w.b == last_from) {
            // the bin was requested and still overflowed the census: once more alone
            if (alone) {
                w_io = w;
                return W_NEED;
            }
            alone = true;
            if (tid < kNB / 32u) e_req()[tid] = 0u;
            TSM_LDS_SYNC();
            if (tid == 0) set_bit(e_req(), w.b);
            TSM_LDS_SYNC();
        } else {
            alone = false;
            // a walk with ties down is followed by one with ties up: its
            // needs before w.b come too
            if (K == FK_R) replan_draw(w.x, w.x, w.b, bend);
            request_round(K, w.b, draw, acc_next, kB == 0, kB == 1);
        }
        last_from = w.b;
        census_clear();
        eng_pass<EP_CENSUS>(f, q, vb, 0.0f);
        census_finish(vb, f.m.t);
    }
}

// Fold K's two bound walks at once: ties down (kB 1) on wave 0 from wl, ties
// up (kB 2) on wave 1 from wh, with shared census rounds wherever either
// lacks a bin.  The walks read the same sums and census and write their own
// bin-start records (e_sstart, e_shi; e_pstart gets the same positions from
// both).  Sets *rl and *rh; returns W_NEED when a bin holds more distinct
// values than the census, else W_DONE.  A census round for one walk replaces
// the runs the other has decided by: its run is then kNoRun, and the caller
// finds it again (locate) from its bin and position.
constexpr uint32_t kSc2 = 16;  // e_sc() words 16..27: the two walks' results, 6 words each
template <int K>
__device__ __noinline__ uint32_t run_walk2(Fin& f_in, const Filt& q_in, const FBins& vb_in, Walk& wl_io,
                                           Walk& wh_io, uint32_t* rl, uint32_t* rh, uint32_t bend, float T,
                                           float thr, uint32_t force, uint32_t lim, bool draw, bool acc_next) {
    Fin f = f_in;  // a private copy: its fields stay in registers across LDS atomics
    const Filt q = q_in;
    const FBins vb = vb_in;
    const uint32_t tid = threadIdx.x, wid = tid / kWave;
    Walk w0 = wl_io, w1 = wh_io;
    uint32_t r0 = W_NEED, r1 = W_NEED;
    uint32_t from0 = kNoBin, from1 = kNoBin;  // the bin each walk last asked the census for
    bool alone = false;
    for (;;) {
        if (wid < 2u && (wid == 0u ? r0 : r1) == W_NEED) {
            Walk w = wid == 0u ? w0 : w1;
            const uint32_t res = wid == 0u ? walk_bins<K, 1>(w, bend, T, thr, force, lim)
                                           : walk_bins<K, 2>(w, bend, T, thr, force, lim);
            if (lane_id() == 0) {
                uint32_t* o = e_sc() + kSc2 + 6u * wid;
                o[0] = res;
                o[1] = w.b;
                o[2] = w.pos;
                o[3] = w.run;
                o[4] = w.within;
                o[5] = __float_as_uint(w.x);
            }
        }
        TSM_LDS_SYNC();
#pragma unroll
        for (uint32_t j = 0; j < 2u; j++) {
            if ((j == 0u ? r0 : r1) != W_NEED) continue;
            const uint32_t* o = e_sc() + kSc2 + 6u * j;
            Walk& w = j == 0u ? w0 : w1;
            w.b = o[1];
            w.pos = o[2];
            w.run = o[3];
            w.within = o[4];
            w.x = __uint_as_float(o[5]);
            if (j == 0u) r0 = o[0];
            else r1 = o[0];
        }
        TSM_LDS_SYNC();
        if (r0 != W_NEED && r1 != W_NEED) break;
        // a census round from the lower of the bins the walks stopped at; a
        // walk that stops again at the bin it last asked for gets that bin
        // alone, once
        const bool n0 = r0 == W_NEED, n1 = r1 == W_NEED;
        const uint32_t b = n0 && n1 ? min(w0.b, w1.b) : (n0 ? w0.b : w1.b);
        const bool again = (n0 && w0.b == b && from0 == b) || (n1 && w1.b == b && from1 == b);
        if (again) {
            if (alone) {
                wl_io = w0;
                wh_io = w1;
                *rl = r0;
                *rh = r1;
                return W_NEED;
            }
            alone = true;
            if (tid < kNB / 32u) e_req()[tid] = 0u;
            TSM_LDS_SYNC();
            if (tid == 0) set_bit(e_req(), b);
            TSM_LDS_SYNC();
        } else {
            alone = false;
            if (K == FK_R) {
                const float x = n0 && w0.b == b ? w0.x : w1.x, y = n1 && w1.b == b ? w1.x : x;
                replan_draw(fminf(x, y), fmaxf(x, y), b, bend);
            }
            request_round(K, b, draw, acc_next, false, true);
        }
        if (n0 && w0.b == b) from0 = b;
        if (n1 && w1.b == b) from1 = b;
        if (!n0) w0.run = kNoRun;
        if (!n1) w1.run = kNoRun;
        census_clear();
        eng_pass<EP_CENSUS>(f, q, vb, 0.0f);
        census_finish(vb, f.m.t);
    }
    wl_io = w0;
    wh_io = w1;
    *rl = r0;
    *rh = r1;
    return W_DONE;
}

// Has the census hold bin b, by a round for it alone when the current one does
// not; false when the bin holds more distinct values than the census.
__device__ __noinline__ bool census_bin(Fin& f, const Filt& q, const FBins& vb, uint32_t b) {
    if (bit_of(e_cpl(), b)) return true;
    const uint32_t tid = threadIdx.x;
    TSM_LDS_SYNC();  // every thread has seen that the bin is missing
    if (tid < kNB / 32u) e_req()[tid] = b / 32u == tid ? 1u << (b & 31u) : 0u;
    TSM_LDS_SYNC();
    census_clear();
    eng_pass<EP_CENSUS>(f, q, vb, 0.0f);
    census_finish(vb, f.m.t);
    return bit_of(e_cpl(), b);
}

// The candidate at position pos (0-based) of the list, in bin lb: its run and
// index within the run, from the bin's runs.
__device__ __forceinline__ bool locate(uint32_t lb, uint32_t pos, uint32_t* run, uint32_t* within) {
    uint32_t r0, r1;
    runs_of(lb, &r0, &r1);
    uint32_t at = e_pstart()[lb];
    for (uint32_t j = r0; j < r1; j++) {
        const uint32_t m = e_hcnt()[j];
        if (pos < at + m) {
            *run = j;
            *within = pos - at;
            return true;
        }
        at += m;
    }
    return false;
}

constexpr uint32_t kHot = 32;  // weight factor of coarse bins where a fold steps value by value
constexpr uint32_t kFineCap = 1024;  // candidates a fine bin's share of the weight may hold

// Does this thread's coarse bin k hold a predicted event: total crossing a
// power of two, acc = total / tot crossing one, top-p's decision, or the
// draw's r crossing one or reaching zero?  The margins cover the gap between these estimates and the
// f32 folds.
__device__ __forceinline__ bool coarse_hot(const FoldView& w, int k, float u, bool topp, bool draw, float top_p) {
    if (w.ms[k] <= 0.0 && w.mr[k] <= 0.0) return false;
    const double lo = w.S[k] * (1.0 - kPlanEps), hi = (w.S[k] + w.ms[k]) * (1.0 + kPlanEps);
    if (!(lo > 0.0) || binade_of(static_cast<float>(lo)) != binade_of(static_cast<float>(hi))) return true;
    if (topp) {
        // acc stops at top_p: a bin that starts past it is never walked by acc
        const double tp = static_cast<double>(top_p) * w.tot;
        if (lo <= tp * (1.0 + kPlanEps)) {
            if (binade_of(static_cast<float>(lo / w.tot)) != binade_of(static_cast<float>(hi / w.tot))) return true;
            if (tp <= hi) return true;
        }
    }
    if (draw) {
        const double r0 = static_cast<double>(u) * w.kept, eps = kPlanEps * r0;
        const double rhi = r0 - w.R[k] + eps, rlo = r0 - (w.R[k] + w.mr[k]) - eps;
        if (rhi > 0.0 && (!(rlo > 0.0) || binade_of(static_cast<float>(rlo)) != binade_of(static_cast<float>(rhi))))
            return true;
    }
    return false;
}

// The last bin at or before `limit` where total's walks with ties down and up
// start from the same value: from there on that value is total's own.
__device__ uint32_t last_agree(uint32_t limit) {
    const uint32_t tid = threadIdx.x;
    if (tid == 0) e_sc()[SC_LAST] = 0u;
    TSM_LDS_SYNC();
    for (uint32_t b = tid; b <= limit && b < kNB; b += kBlock)
        if (__float_as_uint(e_sstart()[b]) == __float_as_uint(e_shi()[b])) atomicMax(&e_sc()[SC_LAST], b);
    TSM_LDS_SYNC();
    const uint32_t r = e_sc()[SC_LAST];
    TSM_LDS_SYNC();
    return r;
}

// After the fine layout's histogram: the coarse bins (this thread's two,
// with cnt0 / cnt1 candidates) holding a part of a fine bin with more
// candidates than a census round takes are crowded; up to kCrowd of them get
// a sub-histogram (one more pass) and are laid out from it (FBins).  Returns
// whether any was, so that the caller counts the fine bins again.
__device__ __noinline__ bool crowd_layout(Fin& f, const Filt& q, FBins& vb, uint32_t cnt0, uint32_t cnt1) {
    const uint32_t tid = threadIdx.x;
    if (tid == 0) e_crowd()[0] = 0u;
    TSM_LDS_SYNC();
#pragma unroll
    for (uint32_t k = 0; k < 2u; k++) {
        const uint32_t c = 2u * tid + k;
        if ((k == 0u ? cnt0 : cnt1) <= kReqCnt / 4u) continue;  // too few to crowd a fine bin
        const uint32_t l0 = e_lay()[c], l1 = e_lay()[c + 1u];
        const uint32_t f0 = min(static_cast<uint32_t>(static_cast<float>(l0) * vb.scale), kNB - 1u);
        const uint32_t f1 = min(static_cast<uint32_t>(static_cast<float>(l1) * vb.scale), kNB - 1u);
        bool crowded = false;
        for (uint32_t j = f0; j <= f1 && !crowded; j++) crowded = e_cnt()[j] > kReqCnt;
        if (crowded) {
            const uint32_t sl = atomicAdd(&e_crowd()[0], 1u);
            if (sl < kCrowd) e_crowd()[1u + sl] = c;
        }
    }
    TSM_LDS_SYNC();
    const uint32_t nc = min(e_crowd()[0], kCrowd);
    if (nc == 0u) return false;
#pragma unroll
    for (uint32_t sl = 0; sl < kCrowd; sl++) vb.cr[sl] = sl < nc ? e_crowd()[1u + sl] : kNoBin;
    // the sub-histograms (by the coarse bins and fr only), then each crowded
    // bin's cumulative counts at its sub-bin edges, wave sl for slot sl
    eng_pass<EP_SUB>(f, q, vb, 0.0f);
    const uint32_t wid = tid / kWave, lane = lane_id();
    if (wid < nc) {
        constexpr uint32_t kPerLane = kSub / kWave;
        static_assert(kPerLane * kWave == kSub, "sub-bins per lane");
        uint32_t h[kPerLane], sum = 0;
#pragma unroll
        for (uint32_t i = 0; i < kPerLane; i++) {
            h[i] = e_hkey()[wid * kSub + lane * kPerLane + i];
            sum += h[i];
        }
        const uint32_t incl = wave_incl_scan(sum);
        const uint32_t n = wave_read(incl, kWave - 1u);
        uint16_t* F = e_cdf(wid);
        uint32_t cum = incl - sum;
#pragma unroll
        for (uint32_t i = 0; i < kPerLane; i++) {
            const uint32_t j = lane * kPerLane + i;
            F[j] = static_cast<uint16_t>(n ? (static_cast<uint64_t>(cum) * 65535u) / n : (j * 65535u) / kSub);
            cum += h[i];
        }
        if (lane == 0) F[kSub] = 65535u;
    }
    TSM_LDS_SYNC();
    return true;
}

// Sampler::distribution (sampler.rs:102-116) for a kept set of `keep`
// candidates (filter q, `len` candidates before the kept count): the first
// min(keep, stride) of them, best first, as (id, p_j / mass), written in
// chunks of up to kExactCap entries, each selected above the previous one's
// last composite, gathered and sorted.  Returns the best id (0 when nothing
// was written).
__device__ __noinline__ uint32_t write_dist_chunks(Fin& f, const Filt& q, uint32_t len, uint32_t keep,
                                                   const DistOut* dist, float y0, float t, float mass) {
    const uint32_t tid = threadIdx.x;
    const uint32_t k = min(keep, dist->stride);
    uint32_t done = 0, best = 0;
    uint64_t last = 0;
    while (done < k) {
        const uint32_t c = min(k - done, kExactCap);
        Filt qd = q;
        if (done) {
            qd.use_min = true;
            qd.min_comp = last;
        }
        if (done + c < len) {
            qd.use_max = true;
            qd.max_comp = select_kth(f, qd, c);
        }
        const uint32_t g = gather_pass(f, qd, kExactCap);
        if (g == 0u) break;
        sort_gathered(f, g);
        last = f.gcomp()[g - 1u];
        if (done == 0u) best = f.rid()[0];
        for (uint32_t j = tid; j < g; j += kBlock) {
            dist->ids[done + j] = f.rid()[j];
            dist->probs[done + j] = glibc_expf((f.ry()[j] - y0) / t) / mass;
        }
        done += g;
        TSM_LDS_SYNC();  // every thread has read gcomp before the next chunk's passes
    }
    if (keep > done && tid == 0) atomicOr(dist->status, TSM_STATUS_DIST_TRUNCATED);
    return best;
}

struct BigOut {
    Pick pick;
    bool small;  // at most kExactCap candidates: the caller finishes them exactly
};

// Rows with a nucleus larger than kExactCap (filter q, best value y0, the
// row's smallest value mlo): total, top-p, the kept mass and the draw by the
// reference's f32 folds.  q1 is q before min-p (min-p keeps at least the
// best candidate).
__device__ __noinline__ BigOut big_nucleus(Fin& f_in, const Filt& q_in, float y0, float mlo, float u,
                                           const DistOut* dist) {
    Fin f = f_in;  // a private copy: its fields stay in registers across LDS atomics
    const Filt q = q_in;
    const uint32_t tid = threadIdx.x;
    const float t = f.m.t;
    const bool topp = !(f.P.top_p >= 1.0f);
    const bool draw = dist == nullptr;
    BigOut out;
    out.small = false;
    out.pick.token = 0xFFFFFFFFu;
    out.pick.keep = 0;
    out.pick.prob = 0.0f;
    out.pick.mass = 0.0f;
    if (tid < 32u) e_exptab()[tid] = kExp2Tab[tid];
    TSM_LDS_SYNC();
    FBins vb;
    vb.vb.y0 = y0;
#pragma unroll
    for (uint32_t sl = 0; sl < kCrowd; sl++) vb.cr[sl] = kNoBin;
    {
        float span = fminf(30.5f, (y0 - mlo) / t);
        if (!(span > 0.0f)) span = 1.0f;
        vb.vb.mul = (static_cast<float>(kNB) / span) / t;
    }
    bool degenerate = !__builtin_isfinite(y0) || !(__builtin_isfinite(vb.vb.mul) && vb.vb.mul > 0.0f);
    uint32_t len = 0;
    if (!degenerate) {
        vb.scale = 0.0f;  // fine = coarse
        eng_pass<EP_HIST>(f, q, vb, 0.0f);
        // when the candidates fill under a quarter of the bins, bin them again
        // over their own range
        const uint32_t kmin = e_sc()[SC_CMIN];
        const bool nan1 = e_sc()[SC_NAN] != 0u;
        TSM_LDS_SYNC();  // read before a second histogram resets them
        if (!nan1 && kmin != 0xFFFFFFFFu) {
            const float cmin = key_to_float(kmin);
            if (vb.vb.bin(cmin) < kNB / 4u) {
                const float sp2 = ((y0 - cmin) / t) * 1.001f;
                const float mul2 = (static_cast<float>(kNB) / sp2) / t;
                if (sp2 > 0.0f && __builtin_isfinite(mul2) && mul2 > 0.0f) {
                    vb.vb.mul = mul2;
                    eng_pass<EP_HIST>(f, q, vb, 0.0f);
                }
            }
        }
        degenerate = e_sc()[SC_NAN] != 0u;
        const uint32_t c0 = e_cnt()[2 * tid], c1 = e_cnt()[2 * tid + 1];
        len = block_sum<kBlock>(c0 + c1, f.tmp());
        if (!degenerate && len > kExactCap) {
            // fine bins of about equal weight: a coarse bin weighs its count,
            // kHot times that where a fold is expected to step value by value
            // (a binade crossing of total, acc or r, top-p's decision, the
            // draw's end), so that those stretches are censused in small bins
            const double m0 = e_mass()[2 * tid], m1 = e_mass()[2 * tid + 1];
            const double wide = 1.0 / (static_cast<double>(vb.vb.mul) * t);
            const double mm[2] = {m0, m1};
            const uint32_t cc[2] = {c0, c1};
            const FoldView w = fold_view(f, mm, cc, u, draw, topp, wide);
            const bool h0 = coarse_hot(w, 0, u, topp, draw, f.P.top_p), h1 = coarse_hot(w, 1, u, topp, draw, f.P.top_p);
            // the hot factor, lowered when hot bins hold most candidates so
            // that a fine bin (a 1/kNB share of the weight) holds at most
            // kFineCap candidates, which the census can take
            const uint32_t hc = block_sum<kBlock>((h0 ? c0 : 0u) + (h1 ? c1 : 0u), f.tmp());
            uint32_t hot = kHot;
            if (hc > 0) {
                const uint64_t room = static_cast<uint64_t>(kNB) * kFineCap;
                const uint64_t cold = len - hc;
                const uint64_t k = room > cold ? (room - cold) / hc : 1u;
                hot = static_cast<uint32_t>(k < 1u ? 1u : (k > kHot ? kHot : k));
            }
            const uint32_t w0c = c0 * (h0 ? hot : 1u);
            const uint32_t w1c = c1 * (h1 ? hot : 1u);
            uint32_t wtot;
            const uint32_t W0 = block_excl_scan<kBlock>(w0c + w1c, f.tmp(), &wtot);
            e_lay()[2 * tid] = W0;
            e_lay()[2 * tid + 1] = W0 + w0c;
            if (tid == kBlock - 1) e_lay()[kNB] = W0 + w0c + (kNB - 1u);
            vb.scale = static_cast<float>(kNB) / static_cast<float>(wtot);
            TSM_LDS_SYNC();
            eng_pass<EP_HIST>(f, q, vb, 0.0f);
            if (crowd_layout(f, q, vb, c0, c1)) eng_pass<EP_HIST>(f, q, vb, 0.0f);
        }
        if (!degenerate && len <= kExactCap) {
            out.small = true;
            out.pick.keep = len;
            return out;
        }
    }
    if (degenerate) {
        // NaN everywhere downstream (an infinite best value, or a NaN
        // candidate): total, acc and r are NaN, no step decides, and the
        // reference keeps every candidate and picks the last (sampler.rs:150)
        if (len == 0) len = count_pass(f, q);
        if (len <= kExactCap) {  // exact_finalize carries the NaNs as the reference does
            out.small = true;
            out.pick.keep = len;
            return out;
        }
        const uint64_t last = exact_at(f, q, ~0ull);
        out.pick.keep = len;
        out.pick.token = static_cast<uint32_t>(last);
        out.pick.mass = __uint_as_float(0x7FC00000u);
        out.pick.prob = out.pick.mass;
        if (dist) write_dist_chunks(f, q, len, len, dist, y0, t, out.pick.mass);
        return out;
    }
    // total's (and the draw's) plans, sums and census
    plan_sr(f, u, draw, topp, 1.0 / (static_cast<double>(vb.vb.mul) * t));
    for (uint32_t i = tid; i < 4u * kNB / 32u; i += kBlock) {
        e_tie()[i] = 0u;
        e_tieb()[i] = 0u;
    }
    TSM_LDS_SYNC();
    request_round(FK_S, 0u, draw && !topp, topp, false);  // with top-p the draw's census waits for acc's
    census_clear();
    eng_pass<EP_SR>(f, q, vb, 0.0f);
    census_finish(vb, t);
    Walk w0;
    w0.x = 0.0f;
    w0.b = 0;
    w0.pos = 0;
    w0.run = w0.within = 0;
    // total: with every unresolved tie rounded down, then up; when both give
    // the same value it is total (the fold is monotone in each step), else
    // the ties are censused and stepped exactly
    float T;
    {
        Walk wl = w0, wh = w0;
        uint32_t rl, rh;
        if (run_walk2<FK_S>(f, q, vb, wl, wh, &rl, &rh, kNB, 0.0f, 0.0f, kNoBin, 0xFFFFFFFFu, draw, topp) == W_NEED)
            return out;
        T = wl.x;
        if (__float_as_uint(wl.x) != __float_as_uint(wh.x)) {
            // the exact walk from the last bin where both walks still agree
            const uint32_t ba = last_agree(kNB - 1u);
            Walk we = w0;
            we.x = e_sstart()[ba];
            we.b = ba;
            we.pos = e_pstart()[ba];
            if (run_walk<FK_S>(f, q, vb, we, kNB, 0.0f, 0.0f, kNoBin, 0xFFFFFFFFu, draw, topp) == W_NEED) return out;
            T = we.x;
        }
    }
    // total (sampler.rs:238)
    uint32_t keep = len, kb = kNoBin;
    float mass = T;
    if (topp) {
        plan_a(T, f.P.top_p);
        clear_ties01();
        request_round(FK_A, 0u, draw, false, false);
        census_clear();
        eng_pass<EP_A>(f, q, vb, T);
        census_finish(vb, t);
        // acc the same way: ties down and up at once; the same decision from both
        // is acc's, else the exact walk
        Walk wal = w0, wa = w0;
        uint32_t ral, ra;
        if (run_walk2<FK_A>(f, q, vb, wal, wa, &ral, &ra, kNB, T, f.P.top_p, kNoBin, 0xFFFFFFFFu, draw, false) ==
            W_NEED)
            return out;
        if (ra != ral || (ra == W_DECIDED && wa.pos != wal.pos)) {
            wa = w0;
            ra = run_walk<FK_A>(f, q, vb, wa, kNB, T, f.P.top_p, kNoBin, 0xFFFFFFFFu, draw, false);
            if (ra == W_NEED) return out;
        }
        if (ra == W_DECIDED) {  // acc >= top_p at candidate wa.pos - 1 (sampler.rs:241-243)
            keep = wa.pos;
            kb = wa.b;
            if (__float_as_uint(e_sstart()[kb]) != __float_as_uint(e_shi()[kb])) {
                // total's value at bin kb still depends on a tie: total's sums
                // again (acc's took their slots) and its exact walk
                const uint32_t ba = last_agree(kb);
                request_round(FK_S, ba, false, false, true);
                census_clear();
                eng_pass<EP_SR>(f, q, vb, 0.0f);
                census_finish(vb, t);
                Walk we = w0;
                we.x = e_sstart()[ba];
                we.b = ba;
                we.pos = e_pstart()[ba];
                if (run_walk<FK_S>(f, q, vb, we, kb + 1u, 0.0f, 0.0f, kNoBin, 0xFFFFFFFFu, draw, false) == W_NEED)
                    return out;
            }
            if (!census_bin(f, q, vb, kb)) return out;
            if (tid < kWave) {  // the kept mass: total's fold through the kept part of bin kb
                Walk wm;
                wm.x = e_sstart()[kb];
                wm.b = kb;
                wm.pos = e_pstart()[kb];
                uint32_t r0, r1;
                runs_of(kb, &r0, &r1);
                walk_runs<FK_S>(wm, r0, r1, 0.0f, 0.0f, keep);
                if (tid == 0) e_sc()[SC_X] = __float_as_uint(wm.x);
            }
            TSM_LDS_SYNC();
            mass = __uint_as_float(e_sc()[SC_X]);
            TSM_LDS_SYNC();
        }
    }
    out.pick.keep = keep;
    out.pick.mass = mass;
    if (dist) {  // Sampler::distribution (sampler.rs:102-116): the kept candidates over mass
        out.pick.token = write_dist_chunks(f, q, len, keep, dist, y0, t, mass);
        return out;
    }
    // the draw (sampler.rs:142-150)
    Walk wr;
    wr.x = u * mass;
    wr.b = 0;
    wr.pos = 0;
    wr.run = wr.within = 0;
    const uint32_t bend = kb != kNoBin ? kb + 1u : kNB;
    // the draw with unresolved ties one way and the other at once; the same pick
    // from both is the draw's, else the exact walk
    Walk wrl = wr;
    uint32_t rrl, rr;
    if (run_walk2<FK_R>(f, q, vb, wrl, wr, &rrl, &rr, bend, 0.0f, 0.0f, kb, keep, draw, false) == W_NEED) return out;
    if (rr != rrl || (rr == W_DECIDED && wr.pos != wrl.pos)) {
        wr = wrl;
        wr.x = u * mass;
        wr.b = 0;
        wr.pos = 0;
        rr = run_walk<FK_R>(f, q, vb, wr, bend, 0.0f, 0.0f, kb, keep, draw, false);
    }
    if (rr == W_NEED) return out;
    uint32_t run = wr.run, within = wr.within;
    if (rr != W_DECIDED) {
        // no step reached r <= 0: the last kept candidate
        uint32_t lb = kb;
        if (lb == kNoBin) {
            if (tid == 0) e_sc()[SC_LAST] = 0u;
            TSM_LDS_SYNC();
            for (uint32_t b = tid; b < kNB; b += kBlock)
                if (e_cnt()[b]) atomicMax(&e_sc()[SC_LAST], b);
            TSM_LDS_SYNC();
            lb = e_sc()[SC_LAST];
        }
        if (!census_bin(f, q, vb, lb) || !locate(lb, keep - 1u, &run, &within)) return out;
    } else if (run == kNoRun) {
        if (!census_bin(f, q, vb, wr.b) || !locate(wr.b, wr.pos - 1u, &run, &within)) return out;
    }
    const uint32_t key = e_hkey()[run];
    const uint32_t minid = e_hmin()[run];
    const float p = e_runp()[run];
    TSM_LDS_SYNC();
    // the pick is the (within+1)-th smallest id among the candidates of value key
    out.pick.token = within == 0u ? minid
                                  : static_cast<uint32_t>(exact_at(
                                        f, q, select_from(f, q, within + 1u, 3, static_cast<uint64_t>(~key) << 32, 32)));
    out.pick.prob = p / mass;
    return out;
}

}  // namespace nuc

// Rows without top-k (window > 1024): the cutoff set (sampler.rs:195-208),
// the window rule, truncation to want, min-p, then top-p and the draw, all
// by re-reading the row.  Up to 1024 survivors are finished by exact_finalize;
// larger sets by the value-bin folds above.  Both reproduce the reference's
// f32 arithmetic.
__device__ __noinline__ Pick reread_nucleus(Fin& f, uint32_t nallow, float u, const DistOut* dist) {
    (void)nallow;
    const uint32_t tid = threadIdx.x;
    const RowMode& m = f.m;
    pen_build(f);
    float mall = -INFINITY, mal = -INFINITY, mlo = INFINITY;
    {
        float la = -INFINITY, lb = -INFINITY, lc = INFINITY;
        row_pass(f, [&](uint32_t id, float x, float y) {
            la = fmaxf(la, y);
            lc = fminf(lc, y);
            if (m.constrained && allowed_bit(f, id)) lb = fmaxf(lb, y);
        });
        la = wave_max(la);
        lb = wave_max(lb);
        lc = -wave_max(-lc);
        float* ftmp = reinterpret_cast<float*>(f.miscd() + 8);
        if ((tid & 63) == 0) {
            ftmp[tid / 64] = la;
            ftmp[16 + tid / 64] = lb;
            ftmp[32 + tid / 64] = lc;
        }
        TSM_LDS_SYNC();
        for (int w = 0; w < kBlock / kWave; w++) {
            mall = fmaxf(mall, ftmp[w]);
            mal = fmaxf(mal, ftmp[16 + w]);
            mlo = fminf(mlo, ftmp[32 + w]);
        }
        TSM_LDS_SYNC();
    }
    const float cut = mall - 30.0f * m.t;  // sampler.rs:198-199
    const float y0 = m.constrained ? mal : mall;
    Filt q0;
    q0.order = ORD_TOTAL_Y;
    q0.use_cut = true;
    q0.cut = cut;
    q0.need_allowed = m.constrained;
    uint32_t n0 = 0xFFFFFFFFu;  // not counted
    if (m.constrained) {
        n0 = count_pass(f, q0);
        if (n0 == 0) {  // sampler.rs:211-221: every allowed id, by total_cmp
            q0.use_cut = false;
            n0 = count_pass(f, q0);
        }
    }
    Filt q1 = q0;
    if (m.want < f.n) {  // ranked.truncate(want)
        if (n0 == 0xFFFFFFFFu) n0 = count_pass(f, q0);
        if (n0 > m.want) {
            q1.use_max = true;
            q1.max_comp = select_kth(f, q0, m.want);
        }
    }
    Filt q2 = q1;
    if (f.P.min_p > 0.0f) {  // extension: min-p prefix
        q2.use_minp = true;
        q2.y0 = y0;
        q2.minp = f.P.min_p;
        // p >= min_p  <=>  y >= y0 + t ln(min_p), up to the roundings of the
        // subtraction, the division and expf (below 1e-6 relative): a band of
        // 1e-3 (|y0| + |t ln min_p| + t) on either side holds every value
        // those roundings could put on the other side
        const float a = m.t * logf(f.P.min_p);
        const float band = 1e-3f * (fabsf(y0) + fabsf(a) + m.t);
        q2.minp_lo = (y0 + a) - band;
        q2.minp_hi = (y0 + a) + band;
    }
    const nuc::BigOut bo = nuc::big_nucleus(f, q2, y0, mlo, u, dist);
    if (!bo.small) return bo.pick;
    if (bo.pick.keep == 0) {  // min-p left nothing: the best candidate alone
        q2 = q1;
        q2.use_max = true;
        q2.max_comp = select_kth(f, q1, 1);
    }
    return nucleus_exact(f, q2, u, dist);
}

}  // namespace tsm
