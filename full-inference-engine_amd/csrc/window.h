// The windowed full-row path: rows whose top-p cut or draw lies past the candidates
// and that no top-k or min-p restricts.
//
// The row's tokens are counted on bins of d = M - y first (no weights), which places
// the cut and the draw to within a few bins.  One pass with exact weights then sums
// the mass above each of the two places and gathers the tokens around them, and the
// exact selection runs on what was gathered.  The counts only say where to look: a
// crossing outside its window is noticed (the exact masses bracket it or do not) and
// the row is taken again around the place those masses give, or by the binned path.
//
// The passes are laid out like k_scan's: one wave per 2048-token tile, 32 tokens a
// lane, no barrier inside a pass.  The count is bound by its one LDS atomic a token
// (21 cycles a wave and CU for random bins), the weighing by vector issue.  At vocab
// 151936 a lone row takes 25-30 us to count, 50-75 to weigh and 10-25 to select; a step
// of 48 open bf16 rows 194 us and one of 1024 flat rows 490, where the single weighted
// pass it replaces (three LDS atomics and a 128-bit product a token, and radix levels
// where a bin overflowed) took 1783 and 752.
#pragma once

// (included by finish.h, whose shared-memory layout and selections it uses)

namespace fie {

// Bins of the count: the top bits of the float d + 1, so 2^kWinOct bins to each
// octave: 1/512 wide at the row's maximum, 1/32 at d = 31, past which every share of
// the mass is below e^-31.  Bin 0 takes what rounding pushes below d = 0.  A bin holds
// its tokens' count (high word) and the sum of the kWinSubs bits of d + 1 below the
// bin's own (all but the last one: a bin may hold every token of the row), so that its
// mass is taken at its tokens' mean d: 16-bit logits put thousands of tokens at one place
// in a bin, and taking its middle was off by 10^-3 of the row's mass.
constexpr int kWinOct = 9, kWinOctaves = 5;
constexpr int kWinShift = 23 - kWinOct, kWinSubs = kWinShift - 1;
static_assert((uint64_t)kMaxTiles * kTile * ((1u << kWinSubs) - 1) < 1ull << 32, "a bin's sum stays in its word");
constexpr uint32_t kWinOrg = (0x3F800000u >> kWinShift) - 1;
constexpr int kWinBins = kWinOctaves * (1 << kWinOct) + 1;
// What is added to d: one, and a shift that keeps the bins' edges off the multiples of
// powers of two (and of those over common temperatures) that 16-bit logits lie on.
constexpr float kWinOne = 1.000337f;
constexpr int kSubBits = 12, kSubBins = 1 << kSubBits;   // bins of a refining count
constexpr int kWinSplit = kGCap / 2;       // a window with more tokens is narrowed to one bin
constexpr int kIdxBits = 19;               // token indexes are below 2^19
constexpr uint32_t kIdxMask = (1u << kIdxBits) - 1;
static_assert(kMaxTiles * kTile <= 1 << kIdxBits, "index bits of a packed composite");
static_assert(2 * kSubBins <= 2 * kGCap && kWinBins <= kGCap, "counts fit the candidate area");

// Rank composites with the index's constant bits left out, so that a window of a few
// thousand keys spans few enough values for one or two refining counts to settle it.
FIE_DEV uint64_t pack_comp(uint32_t key, uint32_t idx) { return ((uint64_t)key << kIdxBits) | (kIdxMask - idx); }
FIE_DEV uint64_t pack_of(uint64_t comp) { return ((comp >> 32) << kIdxBits) | ((uint32_t)comp & kIdxMask); }
FIE_DEV uint32_t pack_key(uint64_t c) { return (uint32_t)(c >> kIdxBits); }
FIE_DEV uint32_t pack_idx(uint64_t c) { return kIdxMask - ((uint32_t)c & kIdxMask); }
FIE_DEV uint64_t unpack_comp(uint64_t c) { return comp_key(pack_key(c), pack_idx(c)); }

// The value of a key as the upper end of a range: the key just below +0 is that of -0,
// which no token has and which compares equal to +0.
FIE_DEV float key_upper(uint32_t k) { return key_to_float(k == 0x7FFFFFFFu ? 0x7FFFFFFEu : k); }

// One count's word of bin j of window k (-1: the whole row's count).
FIE_DEV uint32_t win_count(const FinSmem& S, int k, int j)
{
    return k < 0 ? (uint32_t)(S.cand[j] >> 32) : ((const uint32_t*)S.cand)[k * kSubBins + kSubBins - 1 - j];
}

// Its mass, in units of the row maximum's weight: at the mean d of its tokens, or at
// the middle of a refining count's bin (all of a window's tokens are nearly alike).
FIE_DEV float win_mass(const FinSmem& S, const Win& w, int k, int j, float M)
{
    const uint32_t c = win_count(S, k, j);
    if (c == 0) return 0.0f;
    float y;
    if (k < 0) {
        const uint32_t mean = (uint32_t)(2.0f * ((float)(uint32_t)S.cand[j] / (float)c));
        y = kWinOne - __uint_as_float(((uint32_t)(j + (int)kWinOrg) << kWinShift) + mean);
        return (float)c * __expf(y);
    }
    if (w.byidx) y = w.yh;
    else y = key_to_float(pack_key(w.lo + ((uint64_t)(kSubBins - 1 - j) << w.sh) + ((1ull << w.sh) >> 1)));
    return (float)c * __expf(y - M);
}

// Narrows window k to the bins, in rank order, that the running mass meets between f -
// eps and f + eps: the whole count's bins, or (sub) its own finer ones.  Where those
// hold too many tokens, to the one bin that f lies in: two neighbouring values shared
// by thousands each could not be told apart by a finer count of both.  False when the
// mass does not get there.
FIE_DEV bool win_pick(FinSmem& S, int k, bool sub, bool pen, float M, float f, float eps)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nb = sub ? kSubBins : kWinBins, per = (nb + kFinThreads - 1) / kFinThreads;
    const int ks = sub ? k : -1;
    const Win w = S.win[k];
    const int j0 = min(tid * per, nb), j1 = min(j0 + per, nb);
    float ms = 0.0f;
    uint32_t cs = 0;
    for (int j = j0; j < j1; ++j) {
        ms += win_mass(S, w, ks, j, M);
        cs += win_count(S, ks, j);
    }
    const float mi = wave_incl_scan_f32(ms);
    uint32_t call;
    const uint32_t ce = dwave_excl_scan_u32(cs, &call);
    if (lane == 63) {
        S.red32[wave] = __float_as_uint(mi);
        S.red32[8 + wave] = call;
    }
    __syncthreads();
    float mb = sub ? w.above : 0.0f;
    uint32_t cb = ce;
    for (int v = 0; v < wave; ++v) {
        mb += __uint_as_float(S.red32[v]);
        cb += S.red32[8 + v];
    }
    mb += mi - ms;
    bool found;
    int l, h;
    float above;
    for (;;) {
        // the first bins whose running mass exceeds f - eps, and f + eps (the last bin
        // when none does)
        if (tid == 0) {
            S.wjl = nb;
            S.wjh = nb - 1;
            S.wcl = S.wch = 0;
        }
        __syncthreads();
        if (cs) {
            float run = mb;
            int jl = nb, jh = nb;
            for (int j = j0; j < j1; ++j) {
                run += win_mass(S, w, ks, j, M);
                if (run > f - eps && jl == nb) jl = j;
                if (run > f + eps && jh == nb) jh = j;
            }
            if (jl < nb) atomicMin(&S.wjl, jl);
            if (jh < nb) atomicMin(&S.wjh, jh);
        }
        __syncthreads();
        found = S.wjl < nb;
        l = S.wjl;
        h = S.wjh;
        if (found) {
            float run = mb;
            uint32_t crun = cb;
            for (int j = j0; j < j1; ++j) {
                if (j == l) {
                    S.wcl = crun;
                    S.wab = run;
                }
                run += win_mass(S, w, ks, j, M);
                crun += win_count(S, ks, j);
                if (j == h) S.wch = crun;
            }
        }
        __syncthreads();
        above = S.wab;
        const bool wide = found && eps > 0.0f && S.wch - S.wcl > (uint32_t)kWinSplit;
        if (!wide) break;
        eps = 0.0f;
        __syncthreads();
    }
    if (tid == 0 && found) {
        Win v = S.win[k];
        if (sub) {
            // byidx: every token of the window has one key, and the bins are of the index
            const uint64_t lo = w.byidx ? (w.lo >> kIdxBits) << kIdxBits : w.lo;
            const uint64_t top = lo + ((uint64_t)(kSubBins - l) << w.sh) - 1;
            const uint64_t bot = lo + ((uint64_t)(kSubBins - 1 - h) << w.sh);
            v.hi = top < w.hi ? top : w.hi;
            v.lo = bot > w.lo ? bot : w.lo;
            v.byidx = 0;
        } else {
            auto edge = [](int b) { return __uint_as_float((uint32_t)(b + (int)kWinOrg) << kWinShift) - kWinOne; };
            const float yh = l <= 1 ? M : (M - edge(l)) + 0.0f, yl = (M - edge(h + 1)) + 0.0f;
            v.hi = ((uint64_t)fkey(yh) << kIdxBits) | kIdxMask;
            v.lo = (uint64_t)fkey(yl) << kIdxBits;
            // should it be refined: 16-bit logits mostly put one value in a bin, but for
            // a few penalised tokens among them
            v.byidx = pen ? 0 : 1;
        }
        v.n = S.wch - S.wcl;
        v.above = above;
        const uint64_t r = v.hi - v.lo;
        const int bl = r ? 64 - __builtin_clzll(r) : 0;
        v.sh = v.byidx ? kIdxBits - kSubBits : (bl > kSubBits ? bl - kSubBits : 0);
        v.kmin = 0xFFFFFFFFu;
        v.kmax = 0;
        S.win[k] = v;
    }
    __syncthreads();
    return found;
}

// The gathered list: its first kGCap composites in LDS, the rest (16-bit logits: a value
// shared by over 4096 tokens of a 152k vocabulary, which two more counts of the row would
// narrow in 130 us) in the row's candidate slots of the workspace, when those are free.
struct WinList {
    uint64_t* more;
    uint32_t cap;
    FIE_DEV uint64_t get(const FinSmem& S, int i) const { return i < kGCap ? S.cand[i] : more[i - kGCap]; }
    FIE_DEV void put(FinSmem& S, uint32_t at, uint64_t c) const
    {
        if (at < (uint32_t)kGCap) S.cand[at] = c;
        else if (at < cap) more[at - (uint32_t)kGCap] = c;
    }
};

// The gathered composites [0, n) inside the packed range [lo, hi], in rank order:
// the one where the running weight first exceeds g (excl <= g < excl + meas).  Levels
// of kPassBins bins over the range left, until a bin holds one element.
FIE_DEV SelResult win_select(FinSmem& S, const WinList& wl, int n, uint64_t lo, uint64_t hi, u128 g)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    u128 excl = 0;
    // the range they span: thousands may share a key
    uint64_t mn = ~0ull, mx = 0;
    for (int i = tid; i < n; i += kFinThreads) {
        const uint64_t c = pack_of(wl.get(S, i));
        if (c >= lo && c <= hi) {
            mn = c < mn ? c : mn;
            mx = c > mx ? c : mx;
        }
    }
    mn = ~dwave_max_u64(~mn);
    mx = dwave_max_u64(mx);
    if (lane == 0) {
        S.red64[wave] = mn;
        S.red64[kFinThreads / 64 + wave] = mx;
    }
    __syncthreads();
    for (int v = 0; v < kFinThreads / 64; ++v) {
        mn = S.red64[v] < mn ? S.red64[v] : mn;
        mx = S.red64[kFinThreads / 64 + v] > mx ? S.red64[kFinThreads / 64 + v] : mx;
    }
    if (mx == 0) return SelResult{0, 0, 0, 0};
    lo = mn;
    hi = mx;
    for (;;) {
        const uint64_t r = hi - lo;
        const int bl = r ? 64 - __builtin_clzll(r) : 0, sh = bl > 10 ? bl - 10 : 0;
        for (int i = tid; i < kPassBins; i += kFinThreads) {
            S.pc[i] = 0;
            S.pm_lo[i] = 0;
            S.pm_hi[i] = 0;
        }
        if (tid == 0) S.ibin = -1;
        __syncthreads();
        for (int i = tid; i < n; i += kFinThreads) {
            const uint64_t c = pack_of(wl.get(S, i));
            if (c >= lo && c <= hi) {
                const int b = kPassBins - 1 - (int)((c - lo) >> sh);
                atomicAdd(&S.pc[b], 1u);
                bin_add(S, b, comp_weight(S, wl.get(S, i)));
            }
        }
        __syncthreads();
        // two bins a thread; the limbs are summed apart (each below 2^60)
        static_assert(kPassBins == 2 * kFinThreads, "two bins per thread");
        const u128 b0 = bin_mass(S, 2 * tid), b1 = bin_mass(S, 2 * tid + 1);
        const u128 incl = dwave_incl_scan_u128(b0 + b1);
        if (lane == 63) S.red128[wave] = incl;
        __syncthreads();
        u128 run = incl - (b0 + b1);
        for (int v = 0; v < wave; ++v) run += S.red128[v];
        if (run <= g && g < run + b0 + b1) {
            const bool second = g >= run + b0;
            S.ibin = 2 * tid + (second ? 1 : 0);
            S.bex = second ? run + b0 : run;
            S.bme = second ? b1 : b0;
        }
        __syncthreads();
        const int b = S.ibin;
        if (b < 0) return SelResult{0, 0, 0, 0};
        excl += S.bex;
        g -= S.bex;
        const u128 meas = S.bme;
        const uint32_t cnt = S.pc[b];
        lo += (uint64_t)(kPassBins - 1 - b) << sh;
        const uint64_t top = lo + ((1ull << sh) - 1);
        hi = top < hi ? top : hi;
        if (cnt == 1) {
            for (int i = tid; i < n; i += kFinThreads) {
                const uint64_t c = pack_of(wl.get(S, i));
                if (c >= lo && c <= hi) S.bcomp[0] = unpack_comp(c);
            }
            __syncthreads();
            const uint64_t c = S.bcomp[0];
            __syncthreads();
            return SelResult{c, excl, meas, 1};
        }
        __syncthreads();
    }
}

// x / s as every other path computes it: inside Markstein's range by the corrected
// product (s is in it).
FIE_DEV float win_y(float x, float s, float rs)
{
    if (s == 1.0f) return x + 0.0f;
    if (markstein_ok(x)) return div_markstein(x, s, rs) + 0.0f;
    return scaled(x, s);
}

// One pass over the row, a wave per tile: tokens counted per bin (kWinCount), those of
// the windows in `big` per finer bin (kWinSub), or weighed (kWinWeigh): the exact mass
// above each window into m0, m1, the windows' tokens into S.cand.
//
// Penalised tokens, token 0 and those past the row read NaN in x[], which every step
// passes over; the penalised ones follow one a lane, their logits penalised.  Their
// counts come from k_prep's span bucket, or, where that overflowed, from the whole history,
// read once for the eight tiles that the waves hold (48 rows of vocab 151936 with 16384 ids
// 366 us a step, with 60000 750; 1000 and 3560 when each wave read it for its own tile).
// The next tile's loads are in flight while one is processed.
enum { kWinCount, kWinSub, kWinWeigh };

// A value that the optimizer does not know to equal v: it would take 32 tokens'
// compares with v out in front of the branches that share them, and spill the results
// (with the scheduling barriers every eight tokens, 1024 flat rows 514 -> 485 us).
FIE_DEV float opaque(float v)
{
    asm("" : "+v"(v));
    return v;
}

template <int DT>
FIE_DEV void win_pass(FinSmem& S, const KParams& P, int row, int phase, float s, bool pen, float rep, float pres,
                      float freq, float M, float y0, bool has_cut, const WinList& list, u128& m0,
                      u128& m1)
{
    constexpr int EPL = DTy<DT>::EPL, SZ = DTy<DT>::SZ, NL = kEPT / EPL;
    const fie_sampler_args& a = P.a;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int V = a.vocab, NT = P.NT;
    const char* rowp = (const char*)a.logits + (size_t)row * (size_t)a.row_stride * SZ;
    uint32_t* cnt = S.tp.cnt[wave];
    uint32_t* bits = S.tp.bits[wave];
    uint32_t* sub = (uint32_t*)S.cand;
    const float rs = 1.0f / s, off = M + kWinOne;
    const uint32_t use = phase == kWinSub ? S.wbig : (has_cut ? 3u : 1u);      // the windows looked at

    const uint64_t lo0 = uni64(S.win[0].lo), hi0 = uni64(S.win[0].hi);
    const uint64_t lo1 = uni64(S.win[1].lo), hi1 = uni64(S.win[1].hi);

    auto tally = [&](float x, bool ok) {
        // the quotient to one rounding: the bins only locate
        const uint32_t f = __float_as_uint(__builtin_fmaf(x, -rs, off));
        const uint32_t b = (f >> kWinShift) - kWinOrg;
        if (ok && b < (uint32_t)kWinBins)
            atomicAdd((unsigned long long*)&S.cand[b], (1ull << 32) | ((f >> 1) & ((1u << kWinSubs) - 1)));
    };
    // a window's token in a refining count
    uint32_t kmin[2] = {0xFFFFFFFFu, 0xFFFFFFFFu}, kmax[2] = {0, 0};
    auto refine = [&](float y, uint32_t idx, bool ok) {
        const uint32_t key = fkey(y);
        const uint64_t c = pack_comp(key, idx);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint64_t lo = k ? lo1 : lo0, hi = k ? hi1 : hi0;
            if (!((use >> k) & 1u) || !ok || c < lo || c > hi) continue;
            const bool bi = S.win[k].byidx;
            const uint32_t b = bi ? ((uint32_t)c & kIdxMask) >> (kIdxBits - kSubBits) : (uint32_t)((c - lo) >> S.win[k].sh);
            atomicAdd(&sub[k * kSubBins + b], 1u);
            kmin[k] = min(kmin[k], key);
            kmax[k] = max(kmax[k], key);
        }
    };
    // room for `n` tokens of the wave's lanes in the gathered list
    auto room = [&](uint32_t n) -> uint32_t {
        uint32_t tot, base = 0;
        const uint32_t at = dwave_excl_scan_u32(n, &tot);
        if (tot == 0) return 0;
        if (lane == 0) base = atomicAdd(&S.wn, tot);
        return at + (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
    };
    // what a token not summed yet is: above a window, or in one (gathered)
    auto place = [&](float y, uint32_t idx, bool ok) {
        const uint64_t c = pack_comp(fkey(y), idx);
        const bool in = ok && ((c >= lo0 && c <= hi0) || (has_cut && c >= lo1 && c <= hi1));
        const uint32_t at = room(in ? 1u : 0u);
        if (in) list.put(S, at, comp_key(fkey(y), idx));
        if (ok && c > hi0) m0 += weight_of(S, y, idx);
        if (ok && has_cut && c > hi1) m1 += weight_of(S, y, idx);
    };

    constexpr int kGroup = kFinThreads / 64;              // tiles the waves take at a time
    constexpr int kGroupSpans = kGroup / kWavesPerWG;
    static_assert(kGroupSpans == 2, "two spans' id counts per group");
    uint4 nxt[NL];
    uint32_t nnb[kGroupSpans] = {}, nof = 0;
    auto issue = [&](int t) {
        // past the last tile the last one is loaded again, unused: the loads in flight
        // are then the same at every step
        const int tt = t < NT ? t : NT - 1;
        const int lo = tt * kTile;
        if (lo + kTile <= V) {
#pragma unroll
            for (int j = 0; j < NL; ++j) nxt[j] = load16<DT>(rowp + (size_t)(lo + (j * 64 + lane) * EPL) * SZ);
        } else {
#pragma unroll
            for (int j = 0; j < NL; ++j) nxt[j] = load_group<DT>(rowp, lo + (j * 64 + lane) * EPL, V);
        }
        if (pen) {
            const size_t sr = (size_t)row * P.NS + tt / kWavesPerWG;
            // both spans' of the group, so that all waves agree on how to count it
#pragma unroll
            for (int k = 0; k < kGroupSpans; ++k)
                nnb[k] = P.w.nb[(size_t)row * P.NS + min((t - wave) / kWavesPerWG + k, P.NS - 1)];
            nof = P.w.bk[sr * kBucketCap + lane];
        }
    };
    issue(wave);
    for (int t0 = 0; t0 < NT; t0 += kGroup) {
        const int t = t0 + wave;
        const int lo = t * kTile;
        float x[kEPT];
#pragma unroll
        for (int j = 0; j < NL; ++j) {
#pragma unroll
            for (int e = 0; e < EPL; ++e) x[j * EPL + e] = lane_get<DT>(nxt[j], e);
        }
        const uint32_t nb = wave < kWavesPerWG ? nnb[0] : nnb[1], of = nof;
        // the same in every wave: the barriers below depend on it
        const bool whole = __builtin_amdgcn_readfirstlane((int)max(nnb[0], nnb[1])) > kBucketCap;
        issue(t + kGroup);
        uint32_t any = 0;
        if (pen) {
            const int sp = t / kWavesPerWG;
            const uint32_t toff = (uint32_t)(lo - sp * kSpan);
            const size_t sr = (size_t)row * P.NS + sp;
            uint4* z = (uint4*)cnt;
#pragma unroll
            for (int i = 0; i < kTile / 2 / 4 / 64; ++i) z[i * 64 + lane] = make_uint4(0, 0, 0, 0);
            bits[lane] = 0;
            wave_lds_sync();
            auto count = [&](uint32_t o) {
                if (o >= (uint32_t)kTile) return;
                atomicAdd(&cnt[o >> 1], 1u << ((o & 1) * 16));
                atomicOr(&bits[o >> 5], 1u << (o & 31));
            };
            if (whole) {
                // a span's ids ran past its bucket: all the waves read the whole history once
                // for their tiles together, four ids a thread in flight
                __syncthreads();
                const int64_t h0 = a.hist_offsets[row], h1 = hist_end(a, row);
                for (int64_t h = h0 + tid; h < h1; h += 4 * kFinThreads) {
                    uint32_t id[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        id[k] = h + k * kFinThreads < h1 ? (uint32_t)a.hist_ids[h + k * kFinThreads] : 0u;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint32_t o = id[k] - (uint32_t)(t0 * kTile);
                        if (id[k] == 0 || id[k] >= (uint32_t)V || o >= (uint32_t)(kGroup * kTile)) continue;
                        const uint32_t w = o / kTile, ot = o % kTile;
                        atomicAdd(&S.tp.cnt[w][ot >> 1], 1u << ((ot & 1) * 16));
                        atomicOr(&S.tp.bits[w][ot >> 5], 1u << (ot & 31));
                    }
                }
                __syncthreads();
            } else if (t < NT) {
                if ((uint32_t)lane < nb) count(of - toff);
                for (uint32_t i = lane + 64; i < nb; i += 64) count((uint32_t)P.w.bk[sr * kBucketCap + i] - toff);
            }
            wave_lds_sync();
            any = bits[lane];
            if (__ballot(any != 0) != 0) {
                uint32_t mine = 0;
#pragma unroll
                for (int j = 0; j < NL; ++j) {
                    const int o = (j * 64 + lane) * EPL;
                    mine |= ((bits[o >> 5] >> (o & 31)) & ((1u << EPL) - 1)) << (j * EPL);
                }
#pragma unroll
                for (int i = 0; i < kEPT; ++i)
                    x[i] = __int_as_float(__float_as_int(x[i]) |
                                          (__builtin_amdgcn_sbfe((int)mine, (unsigned)i, 1u) & 0x7FC00000));
            }
        }
        if (t >= NT) continue;                            // past the row: counted with the others, no more
        if (t == 0 && lane == 0) x[0] = __builtin_nanf("");
        if (lo + kTile > V) {
#pragma unroll
            for (int i = 0; i < kEPT; ++i)
                if (elem_index<EPL>(lo, lane, i) >= V) x[i] = __builtin_nanf("");
        }
        if (phase == kWinCount) {
#pragma unroll
            for (int i = 0; i < kEPT; ++i) tally(x[i], true);
        } else {
            // the scaled logits in place of the logits
            if (s != 1.0f) {
                if (DT == FIE_F16 || tile_markstein<DT>(x)) {
#pragma unroll
                    for (int i = 0; i < kEPT; ++i) x[i] = div_markstein(x[i], s, rs);
                } else {
#pragma unroll
                    for (int i = 0; i < kEPT; ++i) x[i] = scaled(x[i], s);
                }
            }
            // A window's ends against this tile's indexes: the end keys' tokens are all
            // in the window, or all outside, unless an end's index lies in the tile
            // (mixed: each token is compared by composite).  ya: above the window from
            // past this value on; [yl, yu]: in it.
            bool mixed = false;
            float ya[2], yl[2], yu[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint64_t wl = k ? lo1 : lo0, wh = k ? hi1 : hi0;
                uint32_t kh = pack_key(wh), kl = pack_key(wl);
                const int ih = (int)pack_idx(wh), il = (int)pack_idx(wl);
                const bool out = !((use >> k) & 1u);
                if (lo + kTile <= ih) --kh;                        // all above
                else if (lo < ih) mixed |= !out;
                if (lo > il) ++kl;                                 // all below
                else if (lo + kTile - 1 > il) mixed |= !out;
                ya[k] = key_upper(kh);
                yu[k] = ya[k];
                yl[k] = out || kl > kh ? __builtin_nanf("") : key_to_float(kl);
            }
            const float a0t = ya[0], a1t = ya[1], l0 = yl[0], u0 = yu[0], l1 = yl[1], u1 = yu[1];
            uint32_t in = 0;
            if (phase == kWinWeigh) {
                const float mt = S.mt[t + 1];
                const uint64_t ct = S.ct[t + 1];
                WeightSum s0, s1;
                if (has_cut) {
#pragma unroll
                    for (int i = 0; i < kEPT; i += 8) {
                        float v0[8], v1[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            const float wt = weight20(x[i + k] - mt);
                            v0[k] = x[i + k] > a0t ? wt : 0.0f;
                            v1[k] = x[i + k] > a1t ? wt : 0.0f;
                        }
                        s0.add8(v0);
                        s1.add8(v1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    m1 += (u128)s1.total() * ct;
                } else {
                    const float a0u = opaque(a0t);
#pragma unroll
                    for (int i = 0; i < kEPT; i += 8) {
                        float v0[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) v0[k] = x[i + k] > a0u ? weight20(x[i + k] - mt) : 0.0f;
                        s0.add8(v0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                m0 += (u128)s0.total() * ct;
            }
            {
                const float lo0u = opaque(l0), up0u = opaque(u0), lo1u = opaque(l1), up1u = opaque(u1);
#pragma unroll
                for (int i = 0; i < kEPT; ++i) {
                    if (i % 8 == 0) __builtin_amdgcn_sched_barrier(0);
                    in |= ((x[i] >= lo0u && x[i] <= up0u) || (x[i] >= lo1u && x[i] <= up1u)) ? 1u << i : 0u;
                }
            }
            if (phase == kWinSub) {
                while (__ballot(in != 0) != 0) {
                    const uint32_t i = in ? (uint32_t)__builtin_ctz(in) : 0u;
                    refine(pick32(x, i) + 0.0f, (uint32_t)elem_index<EPL>(lo, lane, (int)i), in != 0);
                    in &= in - 1;
                }
            } else if (!mixed) {
                uint32_t at = room((uint32_t)__builtin_popcount(in));
                for (; in; in &= in - 1, ++at) {
                    const uint32_t i = (uint32_t)__builtin_ctz(in);
                    list.put(S, at, comp_key(fkey(pick32(x, i) + 0.0f), (uint32_t)elem_index<EPL>(lo, lane, (int)i)));
                }
            } else {
                // tokens equal to a window's upper end at a lower index are above it, and
                // were not summed
                while (__ballot(in != 0) != 0) {
                    const uint32_t i = in ? (uint32_t)__builtin_ctz(in) : 0u;
                    const float y = pick32(x, i) + 0.0f;
                    const uint32_t idx = (uint32_t)elem_index<EPL>(lo, lane, (int)i);
                    const uint64_t c = pack_comp(fkey(y), idx);
                    const bool ok = in != 0;
                    const bool win = ok && ((c >= lo0 && c <= hi0) || (has_cut && c >= lo1 && c <= hi1));
                    const uint32_t at = room(win ? 1u : 0u);
                    if (win) list.put(S, at, comp_key(fkey(y), idx));
                    if (ok && c > hi0 && !(y > a0t)) m0 += weight_of(S, y, idx);
                    if (ok && has_cut && c > hi1 && !(y > a1t)) m1 += weight_of(S, y, idx);
                    in &= in - 1;
                }
            }
        }
        // the penalised tokens: lane l takes those of the tile's 32-token word l
        while (__ballot(any != 0) != 0) {
            const bool ok = any != 0;
            const uint32_t o = (uint32_t)lane * 32 + (ok ? (uint32_t)__builtin_ctz(any) : 0u);
            any &= any - 1;
            float v = 0.0f;
            if (ok)
                v = penalize(load_elem<DT>(rowp, (uint32_t)lo + o), rep, pres, freq,
                             (cnt[o >> 1] >> ((o & 1) * 16)) & 0xFFFFu);
            if (phase == kWinCount) tally(v, ok);
            else if (phase == kWinSub) refine(win_y(v, s, rs), (uint32_t)lo + o, ok);
            else place(win_y(v, s, rs), (uint32_t)lo + o, ok);
        }
        if (pen) wave_lds_sync();
    }
    if (wave == 0) {
        if (phase == kWinCount) tally(y0 * s, lane == 0);
        else if (phase == kWinSub) refine(y0, 0u, lane == 0);
        else place(y0, 0u, lane == 0);
    }
    if (phase == kWinSub) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const uint32_t mn = dwave_min_u32(kmin[k]), mx = dwave_max_u32(kmax[k]);
            if (lane == 0 && mx) {
                atomicMin(&S.win[k].kmin, mn);
                atomicMax(&S.win[k].kmax, mx);
            }
        }
    }
    __syncthreads();
}

// The row's cut and draw (top_p tp, uniform u, whole-row mass sall) over its whole
// vocabulary.  Returns false when it decided nothing.
template <int DT>
FIE_DEV bool windowed_deep(FinSmem& S, const KParams& P, int row, float s, bool pen, float rep, float pres,
                           float freq, uint32_t k0, float M, float tp, double u, u128 sall,
                           const WinList& list, uint64_t* cut_out, u128* T_out, uint64_t* tok_out)
{
    const int tid = threadIdx.x, lane = tid & 63;
    if (!(s >= 0x1p-30f && s <= 0x1p30f) || !(__builtin_fabsf(M) < 0x1p40f) || sall == 0) return false;
    if (pen && P.a.max_row_hist > 65535) return false;        // 16-bit counts
    const float y0 = key_to_float(k0);
    const bool has_cut = tp < 1.0f;
    const u128 thr = has_cut ? ceil_mul_f32(tp, sall) : sall;
    float tot = 0.0f, fc = 0.0f, fd = 0.0f, eps = 0.0f;
    int phase = kWinCount, attempt = 0, level = 0;
    for (;;) {
        if (phase != kWinWeigh)
            for (int i = tid; i < kGCap; i += kFinThreads) S.cand[i] = 0;
        if (tid == 0) S.wn = 0;
        __syncthreads();
        u128 m0 = 0, m1 = 0;
        win_pass<DT>(S, P, row, phase, s, pen, rep, pres, freq, M, y0, has_cut, list, m0, m1);
        bool lost = false;
        if (phase == kWinWeigh) {
            // the exact selections (rules R3, R4) inside the windows
            m0 = block_sum_u128<kFinThreads>(m0, S.red128);
            if (has_cut) m1 = block_sum_u128<kFinThreads>(m1, S.red128);
            const uint32_t n = S.wn;
            uint64_t cut = 0;
            u128 T = sall, g = 0;
            // A list that ran on into the candidate slots leaves the row without any, so
            // that a finish launched again on the same partials comes here again.
            if (n > (uint32_t)kGCap && list.cap > (uint32_t)kGCap)
                for (int t = tid; t < P.NT; t += kFinThreads) {
                    P.w.ncand[(size_t)row * P.NT + t] = 0;
                    P.w.bound[(size_t)row * P.NT + t] = 0xFFFFFFFFu;
                }
            if (n > list.cap) return false;
            if (has_cut) {
                lost = thr - 1 < m1;
                if (!lost) {
                    const SelResult r = win_select(S, list, (int)n, S.win[1].lo, S.win[1].hi, thr - 1 - m1);
                    lost = !r.found;
                    cut = r.comp;
                    T = m1 + r.excl + r.meas;
                }
            }
            if (!lost) {
                g = floor_mul_f64(u, T);
                lost = g < m0;
                if (!lost) {
                    // the draw is at or above the cut: a kept token precedes every other
                    const SelResult r = win_select(S, list, (int)n, S.win[0].lo, S.win[0].hi, g - m0);
                    if (r.found) {
                        *cut_out = cut;
                        *T_out = T;
                        *tok_out = r.comp;
                        return true;
                    }
                    lost = true;
                }
            }
            if (++attempt > 1) return false;
            // a crossing outside its window: again, from the windows' exact masses
            const double unit = (double)tot / u128_to_double(sall);
            if (has_cut)
                fc = S.win[1].above + (float)((u128_to_double(thr) - u128_to_double(m1)) * unit);
            fd = S.win[0].above + (float)((u128_to_double(floor_mul_f64(u, has_cut ? thr : sall)) - u128_to_double(m0)) * unit);
            eps = tot * 0x1p-16f;
            phase = kWinCount;
        } else {
            if (phase == kWinCount && attempt == 0) {
                // the row's estimated mass, and where in it the cut and the draw lie.
                // Windows reach 2^-14 of it to both sides: the bins' spread about their
                // means and the fp32 sums are off by about 10^-5.
                for (int b = tid; b < kWinBins; b += kFinThreads) tot += win_mass(S, S.win[0], -1, b, M);
#pragma unroll
                for (int m = 32; m > 0; m >>= 1) tot += __shfl_xor(tot, m, 64);
                if (lane == 0) S.red32[tid >> 6] = __float_as_uint(tot);
                __syncthreads();
                tot = 0.0f;
                for (int v = 0; v < kFinThreads / 64; ++v) tot += __uint_as_float(S.red32[v]);
                __syncthreads();
                fc = (float)(u128_to_double(thr) / u128_to_double(sall)) * tot;
                fd = (float)u * fc;
                eps = tot * 0x1p-14f;
            }
            uint32_t big = phase == kWinSub ? S.wbig : (has_cut ? 3u : 1u);
            if (phase == kWinSub) {
                // a window binned by index that turned out to hold several keys: the
                // next count bins what is left of it by composite
                __syncthreads();
                if (tid < 2 && ((big >> tid) & 1u) && S.win[tid].byidx) {
                    Win v = S.win[tid];
                    const uint64_t l = (uint64_t)v.kmin << kIdxBits, h = ((uint64_t)v.kmax << kIdxBits) | kIdxMask;
                    if (v.kmax) {
                        v.lo = l > v.lo ? l : v.lo;
                        v.hi = h < v.hi ? h : v.hi;
                    }
                    v.yh = key_to_float(v.kmax);
                    if (v.kmin != v.kmax) {
                        v.byidx = 0;
                        const uint64_t r = v.hi - v.lo;
                        const int bl = r ? 64 - __builtin_clzll(r) : 0;
                        v.sh = bl > kSubBits ? bl - kSubBits : 0;
                        v.split = 1;
                    }
                    S.win[tid] = v;
                }
                __syncthreads();
            }
#pragma unroll 1
            for (int k = 0; k < (has_cut ? 2 : 1); ++k) {
                if (!((big >> k) & 1u)) continue;
                if (phase == kWinSub && S.win[k].split) continue;
                lost |= !win_pick(S, k, phase == kWinSub, pen, M, k ? fc : fd, eps);
            }
            __syncthreads();
            if (tid < 2) S.win[tid].split = 0;
            if (!lost) {
                // windows with too many tokens are counted again on finer bins of the
                // composite (the larger one first, then both)
                const uint32_t n0 = S.win[0].n, n1 = has_cut ? S.win[1].n : 0u;
                big = n0 + n1 <= list.cap ? 0u
                      : (n0 > list.cap / 2 ? 1u : 0u) | (n1 > list.cap / 2 ? 2u : 0u);
                if (tid == 0) S.wbig = big;
                if (big && ++level > 5) return false;
                phase = big ? kWinSub : kWinWeigh;
            } else {
                return false;
            }
        }
        __syncthreads();
    }
}

}  // namespace fie
