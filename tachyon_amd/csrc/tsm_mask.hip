// tsm_mask.hip - the mask producer: JsonObject's allows() for every token of
// the vocabulary, on the GPU, written as the packed allow-bits that
// sample_kernel and split_kernel consume (tsm_batch.mask).
//
// A workgroup owns 256 consecutive tokens and a group of rows.  It stages its
// tokens' bytes in LDS as byte classes and finds the group's distinct states.
// A wave then takes 64 of the tokens through its share of the states: per
// state, the first byte's class and the plain-text flag decide most tokens
// with one ballot; the (state, token) pairs still open go to a queue of the
// wave's own and are stepped 64 at a time, one pair a lane, through the
// automaton's table (tsm_json.h), so that no lane waits for a neighbour whose
// token was decided at once; a plain token passes as soon as its walk comes to
// a string's text.  The answers are collected in LDS, a word per
// state and 32 tokens, and written to every row of the state at the end.
//
// What bounds it: instruction issue and LDS latency of the table steps, not
// memory (256 rows x 151,936 tokens read 1.5 MB and write 4.9 MB).  Stepping
// each (row, token) pair in place, one token a lane and one row after another,
// took 382 us for 256 rows of random JSON prefixes (about 110 distinct
// states): a wave paid for its longest token and for every branch any of its
// tokens took.  This way takes 34 to 39 us from box to box, about 22 us of it
// VALU issue (13.4 M wave instructions, and 7.1 M scalar, 1.2 M LDS ones); 594
// workgroups leave a few CUs with one more than the others.  Smaller workgroups
// even that out but repeat the tables and the search for equal states: 128
// tokens each took 55 us, four waves to 64 tokens 88 us (where 256 tokens took
// 45, before plain tokens passed in the walk).
//
// A mask set (tsm_json_masks_*) evaluates each distinct state of a call once
// and keeps recent states' masks in device memory: one launch copies the rows
// whose state the set holds, if any (and brings the new states into device
// memory), another evaluates the new states, writing each into its slot and
// into every row in that state.  The host keeps the index (state -> slot, least recently
// used out first), so no lookup waits for the GPU.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <list>
#include <unordered_map>
#include <utility>
#include <vector>

#include "tsm_device.h"
#include "tsm_json.h"

namespace tsm {
namespace mask {

constexpr uint32_t kTok = 256;       // tokens per workgroup
constexpr uint32_t kSplit = 2;       // waves that share 64 tokens, each with its part of the states
constexpr int kMB = static_cast<int>(kTok * kSplit);  // threads per workgroup
constexpr uint32_t kStates = 256;    // states per workgroup at most
constexpr uint32_t kHashed = 2 * kStates;  // slots of the table that finds equal states
// Workgroups a launch aims for, two a CU: a short vocabulary's states go to
// several groups, as many as come nearest to it.  Split states pay the fixed
// part twice and equal ones no longer meet, so a vocabulary of 342 blocks on
// stays whole: 256 rows, one group against two, 151,936 ids (594 blocks) 45
// against 63 us (before plain tokens passed at once), 128,256 (501) 30.7
// against 38.2, 100,352 (392) 30.5 against 37.0, 80,000 (313) 29.9 against 28.5.
constexpr uint32_t kFillGroups = 512;
constexpr uint32_t kStage = 16384;   // LDS bytes for the workgroup's tokens
constexpr uint32_t kWords = kTok / 32;
constexpr uint32_t kQueue = 128;     // a wave's open (state, token) pairs: settled above 64, 64 more at a time
constexpr int kTakeAt = 24;          // free lanes that make a wave take new pairs
constexpr uint32_t kToSlot = 0x80000000u;
constexpr uint32_t kPlain = 0x80000000u;  // a token of text bytes only
constexpr uint32_t kText = 0x80000000u;   // inside a string, no escape pending
constexpr uint32_t kOther = 0x80000000u;  // the first classes of a state the tables do not hold

__constant__ const json::Tables kJson = json::make_tables();

struct JsonMaskArgs {
    const uint8_t* bytes;
    const uint32_t* offsets;
    const uint32_t* special;
    const tsm_json_state* states;
    uint32_t* mask;
    // mask sets: where the states' words go, sorted by state: output o is the
    // mask of state out_state[o], for row out_at[o] or slot out_at[o] &
    // ~kToSlot; state group g's outputs are [out_beg[g], out_beg[g + 1])
    const uint32_t* out_state;
    const uint32_t* out_at;
    const uint32_t* out_beg;
    uint32_t* cache;
    uint32_t slot_words;
    uint32_t n_tokens, usable, mask_stride, nwords, nstates;
    uint32_t per_group;  // states per workgroup, <= kStates
};

// States per workgroup for `n` states over `blocks` token blocks: all of them
// (so that equal ones meet) up to kStates, or split into as many groups as
// bring the launch nearest to kFillGroups workgroups.
inline uint32_t states_per_group(uint32_t n, uint32_t blocks) {
    const uint32_t near = (kFillGroups + blocks / 2u) / blocks;
    const uint32_t want_y = near > 1u ? near : 1u;
    const uint32_t gy = want_y < n ? want_y : n;
    const uint32_t per = (n + gy - 1) / gy;
    return per < kStates ? per : kStates;
}

__device__ __forceinline__ bool same_state(const tsm_json_state& a, const tsm_json_state& b) {
    return a.stack == b.stack && a.depth == b.depth && a.state == b.state && a.aux == b.aux && a.len == b.len &&
           a.whitespace == b.whitespace;
}

// LDS order between the lanes of one wave (LDS operations of a wave complete
// in order; this keeps the compiler from moving them across).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// The lanes below this one in a ballot.
__device__ __forceinline__ uint32_t mbcnt(uint64_t b) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(b >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(b), 0u));
}

// Workgroup (token block, state group).  kSet: a mask set's launch.
template <bool kSet>
__global__ __launch_bounds__(kMB) void json_mask_kernel(JsonMaskArgs a) {
    constexpr uint32_t kWaves = static_cast<uint32_t>(kMB) / kWave;
    alignas(16) __shared__ uint8_t stage[kStage]; // the tokens' byte classes, with kNotText
    __shared__ json::Entry next[json::F_COUNT * json::kClasses];
    __shared__ uint32_t first[json::F_COUNT + 1];
    __shared__ uint8_t cls[256];
    __shared__ tsm_json_state st[kStates];            // the group's states
    __shared__ json::Walk walks[kStates];             // their walks' starts
    __shared__ uint8_t flat[kStates];
    __shared__ uint16_t rep[kStates];                 // the first state equal to the state
    __shared__ uint2 todo[kStates];                   // the states to evaluate: kText | state, classes to start with
    __shared__ uint32_t table[kHashed];
    __shared__ uint32_t wave_n[kStates / kWave];
    __shared__ uint32_t bits[kStates * kWords];
    __shared__ uint32_t tok_off[kTok];                // stage offset | length << 16 | kPlain
    __shared__ uint16_t queue[kWaves][kQueue];
    static_assert(kStage <= 32768u && kStates * kWave <= 65536u, "16-bit offsets and queue entries, a bit beside a length");
    const uint32_t tid = threadIdx.x, lane = lane_id(), wid = tid / kWave;
    const uint32_t t0 = blockIdx.x * kTok;
    const uint32_t lim = a.usable < a.n_tokens ? a.usable : a.n_tokens;  // ids with bytes that count
    const uint32_t tend = t0 + kTok < lim ? t0 + kTok : lim;
    const uint32_t s0 = blockIdx.y * a.per_group;
    const uint32_t ns = a.nstates - s0 < a.per_group ? a.nstates - s0 : a.per_group;
    uint32_t lo = 0, hi = 0;
    if (t0 < tend) {
        lo = a.offsets[t0];
        hi = a.offsets[tend];
    }
    const bool staged = hi >= lo && hi - lo <= kStage;
    for (uint32_t i = tid; i < json::F_COUNT * json::kClasses; i += kMB) next[i] = kJson.next[i];
    if (tid < 256u) cls[tid] = kJson.cls[tid];
    if (tid <= json::F_COUNT) first[tid] = kJson.first[tid];
    if (tid < ns) {
        tsm_json_state s = a.states[s0 + tid];
        const uint32_t f = json::flat_of(s);
        json::forget(&s, f);
        st[tid] = s;
        flat[tid] = static_cast<uint8_t>(f);
        if (f != json::F_OTHER) walks[tid] = json::walk_of(s, f);
    }
    for (uint32_t i = tid; i < kHashed; i += kMB) table[i] = 0xFFFFFFFFu;
    for (uint32_t i = tid; i < ns * kWords; i += kMB) bits[i] = 0u;
    __syncthreads();
    if (staged)
        for (uint32_t k = tid; k < hi - lo; k += kMB) stage[k] = cls[a.bytes[lo + k]];
    // equal states: the first to claim a hash slot stands for the others
    bool lead = false;
    if (tid < ns) {
        uint32_t r = tid;
        const tsm_json_state s = st[tid];
        uint32_t h = s.stack * 0x9E3779B1u;
        h = (h ^ (uint32_t(s.depth) | uint32_t(s.state) << 8 | uint32_t(s.aux) << 16 | uint32_t(s.len) << 24)) * 0x85EBCA6Bu;
        h = (h ^ s.whitespace ^ (h >> 15)) * 0xC2B2AE35u;
        for (h >>= 16;; h++) {  // at most kStates of the kHashed slots fill: ends
            const uint32_t old = atomicCAS(&table[h & (kHashed - 1u)], 0xFFFFFFFFu, tid);
            if (old == 0xFFFFFFFFu) break;
            if (same_state(st[old], s)) {
                r = old;
                break;
            }
        }
        rep[tid] = static_cast<uint16_t>(r);
        lead = r == tid;
    }
    const uint64_t leads = wave_ballot(lead);
    if (wid < kStates / kWave && lane == 0) wave_n[wid] = static_cast<uint32_t>(__popcll(leads));
    __syncthreads();
    uint32_t n = 0;
    {
        uint32_t at = 0;
#pragma unroll
        for (uint32_t w = 0; w < kStates / kWave; w++) {
            if (w < wid) at += wave_n[w];
            n += wave_n[w];
        }
        if (lead) {
            const uint32_t f = flat[tid];
            const bool text = f == json::F_STR || f == json::F_STR + 6u;
            todo[at + mbcnt(leads)] =
                make_uint2(tid | (text ? kText : 0u), first[f]);
        }
    }
    // this lane's token
    const uint32_t tt = (wid / kSplit) * kWave + lane, id = t0 + tt;
    bool has = false, mine = false;
    uint32_t c1 = 0;
    bool plain = false;
    if (id < lim) {
        const uint32_t b0 = a.offsets[id], b1 = a.offsets[id + 1u];
        const bool special = a.special != nullptr && ((a.special[id >> 5] >> (id & 31u)) & 1u);
        has = !special && b1 > b0;
        // a token's bytes lie inside [lo, hi) when the offsets are ordered; a
        // token outside it is read from global memory
        mine = has && staged && b0 >= lo && b1 <= hi;
        if (mine) {
            c1 = stage[b0 - lo] & (json::kClasses - 1u);
            // text only (no '"', no '\\', no control byte): accepted whole
            // inside a string with no escape pending
            uint32_t odd = 0;  // the stage's words that hold the token, four classes each
            for (uint32_t k = (b0 - lo) & ~3u; k < b1 - lo; k += 4u) {
                uint32_t w = *reinterpret_cast<const uint32_t*>(stage + k);
                if (k < b0 - lo) w &= 0xFFFFFFFFu << (8u * (b0 - lo - k));
                if (k + 4u > b1 - lo) w &= 0xFFFFFFFFu >> (8u * (k + 4u - (b1 - lo)));
                odd |= w;
            }
            plain = (odd & (json::kNotText * 0x01010101u)) == 0u;
            if (wid % kSplit == 0) tok_off[tt] = (b0 - lo) | (b1 - b0) << 16 | (plain ? kPlain : 0u);
        } else {
            if (has) c1 = cls[a.bytes[b0]] & (json::kClasses - 1u);
            if (wid % kSplit == 0) tok_off[tt] = 0u;  // no length: stepped from global memory
        }
    }
    __syncthreads();
    // the pair this lane walks: its automaton, the classes still to come (none
    // left: the lane is free), whether its token is plain and where its answer goes
    json::Walk walk = {0u, 0u, 0u};
    uint32_t from = 0, to = 0, text = 0, answer = 0;
    uint32_t open = 0;  // pairs in the queue (wave-uniform)
    // free lanes take the queue's last pairs (state q >> 6, this wave's token q & 63)
    auto take = [&](uint64_t free) {
        const uint32_t k = mbcnt(free);
        if (from == to && k < open) {
            const uint32_t q = queue[wid][open - 1u - k];
            const uint32_t s = q >> 6, t = (wid / kSplit) * kWave + (q & 63u);
            walk = walks[s];
            const uint32_t ol = tok_off[t];
            from = ol & 0xFFFFu;
            to = from + ((ol & ~kPlain) >> 16);
            text = (ol & kPlain) ? uint32_t(json::W_TEXT) : 0u;
            answer = s * kTok + t;
        }
        const uint32_t n = static_cast<uint32_t>(__popcll(free));
        open -= n < open ? n : open;
    };
    // walks until the queue is down to `left` pairs (0: and every walk is done)
    auto settle = [&](uint32_t left) {
        wave_lds_order();
        for (;;) {
            const uint64_t free = wave_ballot(from == to);
            if (open > 0u && __popcll(free) >= kTakeAt) {
                take(free);
                if (open <= left && left > 0u) break;
            } else if (open == 0u && (left > 0u || free == ~0ull)) {
                break;
            }
            if (from != to) {
                const json::Entry e = next[walk.row + (stage[from] & (json::kClasses - 1u))];
                const bool ok = json::step_entry(walk, e);
                from += (e.x / json::W_USED) & 1u;
                // a plain token that has come to a string's text (after an escape,
                // say) passes: stepped to its end, 16 rows of 16,000 ids with a
                // 63-byte token took 20 us, the walk in place before 17
                if (!ok || (e.x & text)) from = to;
                if (ok && from == to) atomicOr(&bits[answer >> 5], 1u << (answer & 31u));
            }
        }
        wave_lds_order();
    };
    const uint32_t start = has ? 1u << c1 : 0u;
    uint2 job = todo[wid % kSplit];
    for (uint32_t k = wid % kSplit; k < n; k += kSplit) {
        const uint32_t s = wave_read(job.x, 0) & ~kText;
        const bool sure = plain && (job.x & kText);
        bool ask = !sure && (job.y & start);
        const bool other = (job.y & kOther) != 0u;
        if (k + kSplit < n) job = todo[k + kSplit];
        const uint64_t by = wave_ballot(sure);
        if (by != 0u && lane < 2u)
            atomicOr(&bits[s * kWords + (wid / kSplit) * 2u + lane], static_cast<uint32_t>(lane ? by >> 32 : by));
        if (ask && (other || !mine)) {  // a state or a token the tables do not hold
            ask = false;
            const uint32_t b0 = a.offsets[id];
            if (json::accepts(st[s], a.bytes + b0, a.offsets[id + 1u] - b0))
                atomicOr(&bits[s * kWords + (tt >> 5)], 1u << (tt & 31u));
        }
        const uint64_t aq = wave_ballot(ask);
        if (aq == 0u) continue;
        if (ask) queue[wid][open + mbcnt(aq)] = static_cast<uint16_t>(s << 6 | lane);
        open += static_cast<uint32_t>(__popcll(aq));
        if (open > kQueue - kWave) settle(kQueue - kWave);
    }
    settle(0u);
    __syncthreads();
    // the words of every row (and slot) in these states
    const uint32_t w = tid % kWords, word = blockIdx.x * kWords + w;
    if (word >= a.nwords) return;
    if (!kSet) {
        for (uint32_t r = tid / kWords; r < ns; r += kMB / kWords)
            a.mask[static_cast<size_t>(s0 + r) * a.mask_stride + word] = bits[rep[r] * kWords + w];
    } else {
        const uint32_t oe = a.out_beg[blockIdx.y + 1u];
        for (uint32_t o = a.out_beg[blockIdx.y] + tid / kWords; o < oe; o += kMB / kWords) {
            const uint32_t v = bits[rep[a.out_state[o] - s0] * kWords + w], at = a.out_at[o];
            if (at & kToSlot) a.cache[static_cast<size_t>(at & ~kToSlot) * a.slot_words + word] = v;
            else a.mask[static_cast<size_t>(at) * a.mask_stride + word] = v;
        }
    }
}

// Rows whose state the set holds, and the new states' way into device memory
// beside them.
// Workgroup row y < copies copies kCopyWords words of slot copy_slot[y] to row
// copy_row[y]; row y == copies brings stage_words words of the call's staging
// (the new states and their outputs) from mapped host memory, where every
// workgroup of the evaluation would fetch them over the bus, to `local`.
constexpr int kCB = 256;
constexpr uint32_t kCopyWords = 1024;
struct MaskCopyArgs {
    const uint32_t* copy_slot;  // mapped host memory
    const uint32_t* copy_row;
    const uint32_t* cache;
    uint32_t* mask;
    const uint32_t* staging;    // mapped host memory
    uint32_t* local;
    uint32_t copies, slot_words, mask_stride, nwords, stage_words;
};
__global__ __launch_bounds__(kCB) void mask_copy_kernel(MaskCopyArgs a) {
    __shared__ uint32_t at[2];
    if (blockIdx.y == a.copies) {
        for (uint32_t i = blockIdx.x * kCB + threadIdx.x; i < a.stage_words; i += gridDim.x * kCB)
            a.local[i] = a.staging[i];
        return;
    }
    if (threadIdx.x < 2u) at[threadIdx.x] = threadIdx.x ? a.copy_row[blockIdx.y] : a.copy_slot[blockIdx.y];
    __syncthreads();
    const uint32_t* s = a.cache + static_cast<size_t>(at[0]) * a.slot_words;
    uint32_t* d = a.mask + static_cast<size_t>(at[1]) * a.mask_stride;
    const uint32_t w0 = blockIdx.x * kCopyWords + threadIdx.x;
    uint32_t v[kCopyWords / kCB];
#pragma unroll
    for (uint32_t k = 0; k < kCopyWords / kCB; k++) {
        const uint32_t w = w0 + k * kCB;
        v[k] = w < a.nwords ? s[w] : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kCopyWords / kCB; k++) {
        const uint32_t w = w0 + k * kCB;
        if (w < a.nwords) d[w] = v[k];
    }
}

void set_err(char* err, size_t errlen, const char* fmt, ...) {
    if (!err || errlen == 0) return;
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(err, errlen, fmt, ap);
    va_end(ap);
}

const char* vocab_error(const tsm_vocab* vocab) {
    if (!vocab) return "vocab is NULL";
    if (vocab->reserved != 0) return "vocab->reserved must be 0";
    if (vocab->n_tokens > 0 && (!vocab->bytes || !vocab->offsets))
        return "vocab->bytes and vocab->offsets must be set when n_tokens > 0";
    return nullptr;
}

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev) {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        (void)hipSetDevice(dev);
    }
    ~DeviceGuard() {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// A state's identity: its meaningful fields (the padding is left out).
struct Key {
    uint32_t w[3];
    bool operator==(const Key& o) const { return w[0] == o.w[0] && w[1] == o.w[1] && w[2] == o.w[2]; }
};
struct KeyHash {
    size_t operator()(const Key& k) const {
        uint64_t h = 0x9E3779B97F4A7C15ull;
        for (uint32_t x : k.w) h = (h ^ x) * 0xBF58476D1CE4E5B9ull;
        return static_cast<size_t>(h ^ (h >> 31));
    }
};
inline Key key_of(const tsm_json_state& s) {
    Key k;
    k.w[0] = s.stack;
    k.w[1] = uint32_t(s.depth) | uint32_t(s.state) << 8 | uint32_t(s.aux) << 16 | uint32_t(s.len) << 24;
    k.w[2] = s.whitespace;
    return k;
}

// Staging of one call in pinned, mapped host memory, read by the kernels over
// the bus (no upload step).  First what the evaluation reads: the states to
// evaluate, then their outputs (a slot and the rows, per state) and each state
// group's first output; then the row copies.  The copy kernel brings the
// evaluation's part into device memory on its way; a call without row copies
// has no such launch, and the evaluation reads the staging itself (151,936 ids,
// one new state 20.1 -> 17.2 us a call, 256 rows all new 55.1 -> 52.1; a launch
// of its own costs about 3 us, the bus less).  Two halves take the calls in
// turn, so a call only waits for the kernels of the call before the last.
struct Stage {
    tsm_json_state* states;                     // [rows]
    uint32_t *out_beg, *out_state, *out_at;     // [rows + 1], [2 rows], [2 rows]
    uint32_t *copy_slot, *copy_row;             // [rows]
};
inline size_t stage_pad(size_t n) { return (n + 255u) & ~size_t(255); }
inline size_t stage_eval_bytes(uint32_t rows) {
    const size_t r = rows;
    return stage_pad(r * sizeof(tsm_json_state)) + stage_pad((r + 1u) * 4u) + 2u * stage_pad(2u * r * 4u);
}
inline size_t stage_bytes(uint32_t rows) { return stage_eval_bytes(rows) + 2u * stage_pad(static_cast<size_t>(rows) * 4u); }
// The parts for `rows` rows at `base`; the evaluation's are packed for `jobs`
// states and `outs` outputs, so that their used words are contiguous.
inline Stage stage_at(uint8_t* base, uint32_t rows, uint32_t jobs, uint32_t groups, uint32_t outs) {
    Stage s;
    s.states = reinterpret_cast<tsm_json_state*>(base);
    s.out_beg = reinterpret_cast<uint32_t*>(base + static_cast<size_t>(jobs) * sizeof(tsm_json_state));
    s.out_state = s.out_beg + groups + 1u;
    s.out_at = s.out_state + outs;
    s.copy_slot = reinterpret_cast<uint32_t*>(base + stage_eval_bytes(rows));
    s.copy_row = reinterpret_cast<uint32_t*>(base + stage_eval_bytes(rows) + stage_pad(static_cast<size_t>(rows) * 4u));
    return s;
}

}  // namespace mask
}  // namespace tsm

// The mask set behind tsm_json_masks_*: device memory for `capacity` masks
// (one slot per state, least recently used first out), the staging, and the
// host-side index of which state each slot holds.
struct tsm_json_masks {
    int device = 0;
    uint32_t max_rows = 0, capacity = 0, usable = 0, nwords = 0, slot_words = 0;
    uint32_t* cache = nullptr;   // capacity * slot_words words
    uint8_t* hstage = nullptr;   // pinned host memory: 2 halves of stage_bytes(max_rows)
    uint8_t* dstage = nullptr;   // the same memory's device address
    uint8_t* local = nullptr;    // device memory: the evaluation's part of the running call's staging
    size_t half_bytes = 0;
    int half = 0;
    hipEvent_t used[2] = {nullptr, nullptr};  // recorded after the kernels that read each half
    bool pending[2] = {false, false};
    hipEvent_t done = nullptr;
    bool called = false;
    // the vocabulary the slots were evaluated over
    const void* v_bytes = nullptr;
    const void* v_offsets = nullptr;
    const void* v_special = nullptr;
    uint32_t v_n = 0;
    uint64_t call = 0;
    std::unordered_map<tsm::mask::Key, uint32_t, tsm::mask::KeyHash> where;
    std::vector<tsm::mask::Key> slot_key;
    std::vector<uint64_t> slot_call;  // the last call that used the slot; 0 = free
    std::list<uint32_t> lru;          // front: most recently used
    std::vector<std::list<uint32_t>::iterator> lru_at;
    // scratch of a call: the rows of the states to evaluate, and each state's slot
    std::vector<std::pair<uint32_t, uint32_t>> job_rows;
    std::vector<uint32_t> job_slot;

    void flush() {
        where.clear();
        for (auto& c : slot_call) c = 0;
    }
    void touch(uint32_t s) {
        lru.splice(lru.begin(), lru, lru_at[s]);
        slot_call[s] = call;
    }
    // A slot for a new state: a free one, else the least recently used one
    // that this call has not used; -1 when every slot serves this call.
    int take() {
        const uint32_t s = lru.back();
        if (slot_call[s] == call) return -1;
        if (slot_call[s] != 0) where.erase(slot_key[s]);
        touch(s);
        return static_cast<int>(s);
    }
};

extern "C" {

void tsm_json_init(tsm_json_state* s) {
    if (s) tsm::json::init(s);
}

void tsm_json_advance(tsm_json_state* s, const uint8_t* bytes, size_t n) {
    if (!s || (!bytes && n)) return;
    for (size_t i = 0; i < n; i++) (void)tsm::json::step(*s, bytes[i]);  // advance ignores rejections
}

int tsm_json_accepts(const tsm_json_state* s, const uint8_t* bytes, size_t n) {
    if (!s || (!bytes && n)) return 0;
    tsm_json_state c = *s;
    for (size_t i = 0; i < n; i++)
        if (!tsm::json::step(c, bytes[i])) return 0;
    return 1;
}

int tsm_json_is_complete(const tsm_json_state* s) { return s && s->state == tsm::json::JS_DONE ? 1 : 0; }

int tsm_json_mask(void* stream, const tsm_vocab* vocab, const tsm_json_state* states, uint32_t rows,
                  uint32_t usable, uint32_t* mask, uint32_t mask_stride, char* err, size_t errlen) {
    using tsm::mask::set_err;
    if (const char* ve = tsm::mask::vocab_error(vocab)) return set_err(err, errlen, "%s", ve), 1;
    if (!states) return set_err(err, errlen, "states is NULL"), 1;
    if (!mask) return set_err(err, errlen, "mask is NULL"), 1;
    if (rows == 0 || rows > 65535u) return set_err(err, errlen, "rows %u is outside [1, 65535]", rows), 1;
    if (usable == 0 || usable > TSM_MAX_VOCAB)
        return set_err(err, errlen, "usable %u is outside [1, %u]", usable, TSM_MAX_VOCAB), 1;
    const uint32_t nwords = (usable + 31u) / 32u;
    if (mask_stride < nwords)
        return set_err(err, errlen, "mask_stride %u is below ceil(usable / 32) = %u", mask_stride, nwords), 1;
    tsm::mask::JsonMaskArgs a;
    a.bytes = vocab->bytes;
    a.offsets = vocab->offsets;
    a.special = vocab->special;
    a.states = states;
    a.mask = mask;
    a.out_state = a.out_at = a.out_beg = nullptr;
    a.cache = nullptr;
    a.slot_words = 0;
    a.n_tokens = vocab->n_tokens;
    a.usable = usable;
    a.mask_stride = mask_stride;
    a.nwords = nwords;
    a.nstates = rows;
    const uint32_t blocks = (usable + tsm::mask::kTok - 1) / tsm::mask::kTok;
    a.per_group = tsm::mask::states_per_group(rows, blocks);
    const dim3 grid(blocks, (rows + a.per_group - 1) / a.per_group);
    hipLaunchKernelGGL((tsm::mask::json_mask_kernel<false>), grid, dim3(tsm::mask::kMB), 0,
                       static_cast<hipStream_t>(stream), a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_err(err, errlen, "launch failed: %s", hipGetErrorString(e)), 1;
    return 0;
}

void tsm_json_masks_destroy(tsm_json_masks* m) {
    if (!m) return;
    tsm::mask::DeviceGuard g(m->device);
    if (m->done && m->called) (void)hipEventSynchronize(m->done);
    for (int h = 0; h < 2; h++)
        if (m->used[h]) (void)hipEventDestroy(m->used[h]);
    if (m->done) (void)hipEventDestroy(m->done);
    if (m->cache) (void)hipFree(m->cache);
    if (m->local) (void)hipFree(m->local);
    if (m->hstage) (void)hipHostFree(m->hstage);
    delete m;
}

tsm_json_masks* tsm_json_masks_create(int device, uint32_t max_rows, uint32_t capacity, uint32_t usable, char* err,
                                      size_t errlen) {
    using tsm::mask::set_err;
    if (max_rows == 0 || max_rows > 65535u) return set_err(err, errlen, "max_rows %u is outside [1, 65535]", max_rows), nullptr;
    if (capacity > 65536u) return set_err(err, errlen, "capacity %u is above 65536", capacity), nullptr;
    if (usable == 0 || usable > TSM_MAX_VOCAB)
        return set_err(err, errlen, "usable %u is outside [1, %u]", usable, TSM_MAX_VOCAB), nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev)
        return set_err(err, errlen, "device %d is not a visible GPU", device), nullptr;
    tsm::mask::DeviceGuard g(device);
    tsm_json_masks* m = new tsm_json_masks();
    m->device = device;
    m->max_rows = max_rows;
    m->capacity = capacity;
    m->usable = usable;
    m->nwords = (usable + 31u) / 32u;
    m->slot_words = (m->nwords + 63u) & ~63u;  // slots start on 256-byte boundaries
    m->half_bytes = tsm::mask::stage_bytes(max_rows);
    hipError_t e = hipSuccess;
    if (capacity > 0) e = hipMalloc(&m->cache, static_cast<size_t>(capacity) * m->slot_words * 4u);
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void**>(&m->hstage), 2 * m->half_bytes, hipHostMallocMapped);
    if (e == hipSuccess) e = hipHostGetDevicePointer(reinterpret_cast<void**>(&m->dstage), m->hstage, 0);
    if (e == hipSuccess) e = hipMalloc(&m->local, tsm::mask::stage_eval_bytes(max_rows));
    for (int h = 0; h < 2 && e == hipSuccess; h++) e = hipEventCreateWithFlags(&m->used[h], hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&m->done, hipEventDisableTiming);
    if (e != hipSuccess) {
        set_err(err, errlen, "device setup failed: %s", hipGetErrorString(e));
        tsm_json_masks_destroy(m);
        return nullptr;
    }
    m->job_rows.reserve(max_rows);
    m->job_slot.reserve(max_rows);
    m->slot_key.resize(capacity);
    m->slot_call.assign(capacity, 0);
    m->lru_at.resize(capacity);
    for (uint32_t s = 0; s < capacity; s++) m->lru_at[s] = m->lru.insert(m->lru.end(), s);
    return m;
}

void tsm_json_masks_reset(tsm_json_masks* m) {
    if (m) m->flush();
}

int tsm_json_masks_fill(tsm_json_masks* m, void* stream, const tsm_vocab* vocab, const tsm_json_state* states,
                        uint32_t rows, uint32_t* mask, uint32_t mask_stride, tsm_json_fill_stats* stats, char* err,
                        size_t errlen) {
    using tsm::mask::set_err;
    if (!m) return set_err(err, errlen, "mask set is NULL"), 1;
    if (const char* ve = tsm::mask::vocab_error(vocab)) return set_err(err, errlen, "%s", ve), 1;
    if (!states) return set_err(err, errlen, "states is NULL"), 1;
    if (!mask) return set_err(err, errlen, "mask is NULL"), 1;
    if (rows == 0 || rows > m->max_rows)
        return set_err(err, errlen, "rows %u is outside [1, %u] (the set's max_rows)", rows, m->max_rows), 1;
    if (mask_stride < m->nwords)
        return set_err(err, errlen, "mask_stride %u is below ceil(usable / 32) = %u", mask_stride, m->nwords), 1;
    tsm::mask::DeviceGuard g(m->device);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    m->call++;
    if (vocab->bytes != m->v_bytes || vocab->offsets != m->v_offsets || vocab->special != m->v_special ||
        vocab->n_tokens != m->v_n) {
        m->flush();  // the slots hold another vocabulary's masks
        m->v_bytes = vocab->bytes;
        m->v_offsets = vocab->offsets;
        m->v_special = vocab->special;
        m->v_n = vocab->n_tokens;
    }
    const int h = m->half;
    m->half ^= 1;
    if (m->pending[h]) {  // the kernels that last read this half are done
        const hipError_t e = hipEventSynchronize(m->used[h]);
        if (e != hipSuccess) return set_err(err, errlen, "waiting for the staging failed: %s", hipGetErrorString(e)), 1;
        m->pending[h] = false;
    }
    uint8_t* hbase = m->hstage + h * m->half_bytes;
    uint8_t* dbase = m->dstage + h * m->half_bytes;
    // this call's states: the slot that holds each one's mask, or the job that
    // evaluates it
    constexpr uint32_t kJob = 0x80000000u;
    std::unordered_map<tsm::mask::Key, uint32_t, tsm::mask::KeyHash> src;
    src.reserve(rows * 2u);
    m->job_rows.clear();
    m->job_slot.clear();
    // the copies' and states' places do not depend on how many jobs there are
    const tsm::mask::Stage at = tsm::mask::stage_at(hbase, m->max_rows, 0, 0, 0);
    uint32_t jobs = 0, copies = 0, hits = 0, distinct = 0, outs = 0;
    for (uint32_t r = 0; r < rows; r++) {
        const tsm::mask::Key k = tsm::mask::key_of(states[r]);
        uint32_t where;
        const auto seen = src.find(k);
        if (seen != src.end()) {
            where = seen->second;
        } else {
            distinct++;
            const auto cached = m->where.find(k);
            if (cached != m->where.end()) {
                m->touch(cached->second);
                hits++;
                where = cached->second;
            } else {
                tsm_json_state st = states[r];
                std::memset(st.pad, 0, sizeof(st.pad));
                at.states[jobs] = st;
                const int slot = m->capacity ? m->take() : -1;
                if (slot >= 0) {
                    m->slot_key[slot] = k;
                    m->where.emplace(k, static_cast<uint32_t>(slot));
                    outs++;
                }
                m->job_slot.push_back(slot >= 0 ? static_cast<uint32_t>(slot) : kJob);
                where = kJob | jobs++;
            }
            src.emplace(k, where);
        }
        if (where & kJob) {
            m->job_rows.emplace_back(where & ~kJob, r);
            outs++;
        } else {
            at.copy_slot[copies] = where;
            at.copy_row[copies++] = r;
        }
    }
    const uint32_t blocks = (m->usable + tsm::mask::kTok - 1) / tsm::mask::kTok;
    const uint32_t per = jobs ? tsm::mask::states_per_group(jobs, blocks) : 1u;
    const uint32_t groups = (jobs + per - 1) / per;
    uint32_t stage_words = 0;
    if (jobs > 0) {  // the outputs, sorted by state: its slot, then its rows
        const tsm::mask::Stage hs = tsm::mask::stage_at(hbase, m->max_rows, jobs, groups, outs);
        std::vector<uint32_t>& next = m->job_slot;  // becomes each job's next output
        std::sort(m->job_rows.begin(), m->job_rows.end());
        uint32_t o = 0, i = 0;
        for (uint32_t j = 0; j < jobs; j++) {
            if (j % per == 0) hs.out_beg[j / per] = o;
            if (next[j] != kJob) {
                hs.out_state[o] = j;
                hs.out_at[o++] = tsm::mask::kToSlot | next[j];
            }
            for (; i < m->job_rows.size() && m->job_rows[i].first == j; i++) {
                hs.out_state[o] = j;
                hs.out_at[o++] = m->job_rows[i].second;
            }
        }
        hs.out_beg[groups] = o;
        stage_words = jobs * static_cast<uint32_t>(sizeof(tsm_json_state) / 4u) + groups + 1u + 2u * outs;
    }
    const tsm::mask::Stage ds = tsm::mask::stage_at(dbase, m->max_rows, jobs, groups, outs);
    if (copies > 0) {
        tsm::mask::MaskCopyArgs c;
        c.copy_slot = ds.copy_slot;
        c.copy_row = ds.copy_row;
        c.cache = m->cache;
        c.mask = mask;
        c.staging = reinterpret_cast<const uint32_t*>(dbase);
        c.local = reinterpret_cast<uint32_t*>(m->local);
        c.copies = copies;
        c.slot_words = m->slot_words;
        c.mask_stride = mask_stride;
        c.nwords = m->nwords;
        c.stage_words = stage_words;
        const dim3 grid((m->nwords + tsm::mask::kCopyWords - 1) / tsm::mask::kCopyWords, copies + (jobs ? 1u : 0u));
        hipLaunchKernelGGL(tsm::mask::mask_copy_kernel, grid, dim3(tsm::mask::kCB), 0, s, c);
    }
    hipError_t e = hipGetLastError();
    // (a failed copy brought no states: the evaluation would read what the last call left)
    if (e == hipSuccess && jobs > 0) {
        const tsm::mask::Stage ls = copies > 0 ? tsm::mask::stage_at(m->local, m->max_rows, jobs, groups, outs) : ds;
        tsm::mask::JsonMaskArgs a;
        a.bytes = vocab->bytes;
        a.offsets = vocab->offsets;
        a.special = vocab->special;
        a.states = ls.states;
        a.mask = mask;
        a.out_state = ls.out_state;
        a.out_at = ls.out_at;
        a.out_beg = ls.out_beg;
        a.cache = m->cache;
        a.slot_words = m->slot_words;
        a.n_tokens = vocab->n_tokens;
        a.usable = m->usable;
        a.mask_stride = mask_stride;
        a.nwords = m->nwords;
        a.nstates = jobs;
        a.per_group = per;
        hipLaunchKernelGGL((tsm::mask::json_mask_kernel<true>), dim3(blocks, groups), dim3(tsm::mask::kMB), 0, s, a);
    }
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(m->used[h], s);
    if (e == hipSuccess) e = hipEventRecord(m->done, s);
    if (e != hipSuccess) {
        m->flush();  // the index names the call's new states already, whose masks may never be written
        return set_err(err, errlen, "launch failed: %s", hipGetErrorString(e)), 1;
    }
    m->pending[h] = true;
    m->called = true;
    if (stats) {
        stats->rows = rows;
        stats->distinct = distinct;
        stats->hits = hits;
        stats->evaluated = jobs;
    }
    return 0;
}

}  // extern "C"
