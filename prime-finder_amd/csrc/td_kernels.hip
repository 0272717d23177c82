// td_kernels.hip -- Phase-1 trial division for gfx950.
//
// Problem (reference trial_div.cu:46-123, trial_div_cpu.c:32-111): for every
// prime p of a list and every (k, j) of a K x J grid, eliminate (k, j) when
//   p | N      = 10^a - k 10^b - j 10^c - 1,                  or
//   p | rev(N) = 10^a - rev(k) 10^(a-b-lk) - rev(j) 10^(a-c-lj) - 1,
// with the reference CPU sieve's gating (trial_div_cpu.c:41,57-63,68,73,82,97):
// no normal solve when 10^c == 0 (mod p), no rev solve for a k (or j digit
// group) whose exponent is negative or whose power of ten vanishes mod p.
//
// Both conditions are linear in one unknown once the other is fixed, so per
// prime and row k there is one residue u per condition whose small values
// are the hits (u = j - 1 for N, u = rev(j) - 1 for each j digit group).
// Along k these residues move by fixed steps, so after a per-prime setup the
// k loop needs only modular subtractions and compares: no multiplications.
//
// Work split:
//   td_split_kernel        wave-ballot compaction of primes < 2^16 into a
//                          scratch list (one atomic per wave), and input
//                          validation;
//   td_small_setup_kernel  per small prime: the residues and digit-group
//                          constants, with the reference's exact arithmetic
//                          (Fermat inverses, the powmod conventions);
//   td_rows_kernel         small primes hit many j per row, so a workgroup
//                          owns a band of TD_ROWS rows in LDS, lanes spread
//                          over (row, prime), marks are LDS atomics and the
//                          band is OR-ed into HBM once;
//   td_large_kernel        one lane per prime >= 2^16 when the rev
//                          condition's j digit groups do not merge (a-c < D_j):
//                          Montgomery setup, then a k loop of 3-op modular
//                          steps with a rare divergent hit path (global
//                          atomic OR);
//   td_mid_kernel          primes in [2^16, TD_LAT_MIN) with merged groups (one
//                          rev residue per k, see td_hits): the same k loop,
//                          TD_MID_SPLIT lanes per prime over slices of k;
//   td_lattice_kernel      primes >= TD_LAT_MIN with merged groups: each
//                          condition is one residue sequence c0 + t sig mod p,
//                          and its hits are found one by one by a
//                          continued-fraction first-hit search (td_lattice.h)
//                          instead of stepping every k.
#include "pf_hip.h"
#include "td_lattice.h"
#include "../../include/trial_div.h"

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>
#include <vector>

namespace {

constexpr uint32_t TD_SMALL_LIMIT = 1u << 16;   // row kernel below, lane kernel above
constexpr uint32_t TD_SMALL_CAP   = 65536;      // list entries below TD_SMALL_LIMIT
constexpr uint32_t TD_TBL         = 25;         // uint32 fields per small-prime table entry
constexpr uint32_t TD_ROWS        = 4;          // rows per row-kernel workgroup
constexpr uint32_t TD_BLOCK       = 256;
constexpr uint32_t TD_PMAX        = 0x80000000u;
constexpr int      TD_SETUP_GRID  = 32;

// Small-prime table, structure of arrays: field f of entry i lives at
// tbl[f * TD_SMALL_CAP + i], so lanes reading consecutive entries coalesce.
enum {
    TT_P = 0, TT_MAGIC = 1, TT_FLAGS = 2, TT_UN0 = 3, TT_B = 4,
    TT_CM = 5,   // 4 words: Cm[lj-1]
    TT_E = 9,    // 16 words: E[(lk-1)*4 + (lj-1)]
};

// Word-pattern fills (the reference's small-prime Phase 0, sieve_table.c:93-243
// and sieve.c:4-31, done per row on the device): for the odd primes below 32
// other than 5 a 32-bit word of a row holds several hits of each condition,
// so the merged-rev row kernel ORs whole words from per-class masks instead
// of marking hits one by one.  For p >= 32 a period spans more than a word
// and the row kernel's strided marks are already one store per period.
constexpr int      TD_NFILL        = 9;
constexpr uint32_t TD_FILL_CLASSES = 153;   // 3 + 7 + 11 + ... + 31: classes of all fill primes
__constant__ uint32_t c_fill_p[TD_NFILL]   = {3u, 7u, 11u, 13u, 17u, 19u, 23u, 29u, 31u};
__constant__ uint32_t c_fill_off[TD_NFILL] = {0u, 3u, 10u, 21u, 34u, 51u, 70u, 93u, 122u};

// Index of p among the fill primes, or -1.
__host__ __device__ __forceinline__ int td_fill_index(uint32_t p)
{
    switch (p) {
    case 3u: return 0;  case 7u: return 1;  case 11u: return 2; case 13u: return 3;
    case 17u: return 4; case 19u: return 5; case 23u: return 6; case 29u: return 7;
    case 31u: return 8;
    default: return -1;
    }
}

// ctrl words: CT_FILL has bit f set when fill prime f is in the list, and
// CT_FILL_IDX + f is the setup-table entry of (one copy of) that prime.
enum { CT_SMALL_COUNT = 0, CT_ERROR = 1, CT_ITEMS = 2, CT_ITEM_OVF = 3, CT_MID_COUNT = 4,
       CT_FILL = 5, CT_FILL_IDX = 6, CT_WORDS = CT_FILL_IDX + TD_NFILL };

// Class-mask table of the fill primes for a row of J bits (qw = ceil(J/32)
// words per mask): mask (kind, f, r) at word (kind * TD_FILL_CLASSES +
// c_fill_off[f] + r) * qw; kind 0 holds the j with j mod p == r, kind 1 the
// j with R(j) mod p == r (R(j) = rev(j) padded with zeros to D_j digits).
constexpr uint32_t TD_FILL_WORDS = 2u * TD_FILL_CLASSES * ((9999u + 31u) / 32u);

// Primes in [TD_SMALL_LIMIT, mid limit) are compacted into a list of at most
// TD_MID_CAP entries (every prime of [2^16, 2^24) fits) for the split k-loop
// kernel.
constexpr uint32_t TD_MID_CAP = 1100000;

// Row-kernel work items: (small prime, kind, part), each at most TD_CH
// marking steps, so that lanes of one wave get comparable work.
constexpr uint32_t TD_CH       = 32;
constexpr uint32_t TD_ITEM_CAP = 32768;   // > 2 * 6542 + 20000/32 * sum(1/p)
enum { TI_N = 0, TI_REV = 1, TI_WHOLE = 2, TI_ONE = 3 };

__device__ __forceinline__ int td_ndigits(uint32_t x)
{
    return 1 + (x >= 10u) + (x >= 100u) + (x >= 1000u) + (x >= 10000u);
}

// x mod p for x < 2^32 with magic = floor(2^32 / p).
__device__ __forceinline__ uint32_t td_mod(uint32_t x, uint32_t p, uint32_t magic)
{
    uint32_t q = __umulhi(x, magic);
    uint32_t r = x - q * p;
    return r >= p ? r - p : r;
}

// The reference's square-and-multiply (trial_div_cpu.c:22-30) for p < 2^16,
// where every product fits in 32 bits.
__device__ uint32_t td_powmod16(uint32_t base, uint64_t e, uint32_t p)
{
    uint32_t acc = 1u, sq = base % p;
    while (e) {
        if (e & 1u) acc = acc * sq % p;
        sq = sq * sq % p;
        e >>= 1;
    }
    return acc;
}

__global__ void td_reset_kernel(uint32_t *ctrl)
{
    if (threadIdx.x == 0) {
        ctrl[CT_SMALL_COUNT] = 0u;
        ctrl[CT_MID_COUNT] = 0u;
        ctrl[CT_FILL] = 0u;
    }
}

__global__ __launch_bounds__(TD_BLOCK)
void td_split_kernel(const uint32_t *__restrict__ primes, uint32_t n,
                     uint32_t *__restrict__ small, uint32_t *__restrict__ mid, uint32_t mid_hi,
                     uint32_t *__restrict__ ctrl)
{
    const uint32_t i = blockIdx.x * TD_BLOCK + threadIdx.x;
    const uint32_t p = i < n ? primes[i] : TD_PMAX - 1u;
    const bool bad = i < n && (p < 2u || p >= TD_PMAX);
    const bool is_small = !bad && p < TD_SMALL_LIMIT;
    const bool is_mid = !bad && i < n && p >= TD_SMALL_LIMIT && p < mid_hi;
    if (bad) atomicOr(&ctrl[CT_ERROR], 1u);
    const int lane = __lane_id();
    // wave-ballot compaction: one atomic per wave and list
    const uint64_t mask = __ballot(is_small);
    if (mask) {
        const int leader = __ffsll((unsigned long long)mask) - 1;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&ctrl[CT_SMALL_COUNT], (uint32_t)__popcll(mask));
        base = __shfl(base, leader);
        if (is_small) {
            const uint32_t pos = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
            if (pos < TD_SMALL_CAP) small[pos] = p;
            else atomicOr(&ctrl[CT_ERROR], 2u);
        }
    }
    const uint64_t mm = __ballot(is_mid);
    if (mm) {
        const int leader = __ffsll((unsigned long long)mm) - 1;
        uint32_t base = 0;
        if (lane == leader) base = atomicAdd(&ctrl[CT_MID_COUNT], (uint32_t)__popcll(mm));
        base = __shfl(base, leader);
        if (is_mid) {
            const uint32_t pos = base + (uint32_t)__popcll(mm & ((1ull << lane) - 1ull));
            if (pos < TD_MID_CAP) mid[pos] = p;
            else atomicOr(&ctrl[CT_ERROR], 4u);
        }
    }
}

__global__ __launch_bounds__(TD_BLOCK)
void td_small_setup_kernel(const uint32_t *__restrict__ small,
                           uint32_t *__restrict__ ctrl,
                           long long a, long long b, long long c,
                           uint32_t *__restrict__ tbl)
{
    const uint32_t count = min(ctrl[CT_SMALL_COUNT], TD_SMALL_CAP);
    for (uint32_t i = blockIdx.x * TD_BLOCK + threadIdx.x; i < count;
         i += gridDim.x * TD_BLOCK) {
        const uint32_t p = small[i];
        uint32_t *e = tbl + i;          // field f at e[f * TD_SMALL_CAP]
        const uint32_t magic = (uint32_t)(0x100000000ull / p);
        // x y mod p for x, y < p < 2^16 (the product fits 32 bits)
        auto mulm = [&](uint32_t x, uint32_t y) { return td_mod(x * y, p, magic); };
        // The eleven powers of ten a prime needs (10^a, 10^b, 10^c and
        // 10^(a-b-l), 10^(a-c-l) for l = 1..4), sharing their squarings:
        // right to left over the exponents' bits, which are the same in
        // every lane.  These are the residues of the reference's powmod
        // (trial_div_cpu.c:22-30), 10^0 = 1 and p = 2, 5 included; negative
        // exponents are gated below.
        uint64_t ex[11] = {(uint64_t)a, (uint64_t)b, (uint64_t)c};
        for (int l = 1; l <= 4; l++) {
            ex[2 + l] = a - b - l >= 0 ? (uint64_t)(a - b - l) : 0u;
            ex[6 + l] = a - c - l >= 0 ? (uint64_t)(a - c - l) : 0u;
        }
        uint64_t top = 0;
        uint32_t pw[11];
#pragma unroll
        for (int q = 0; q < 11; q++) {
            pw[q] = 1u % p;
            top |= ex[q];
        }
        uint32_t sq = 10u % p;
        for (int bit = 0; (top >> bit) != 0u; bit++) {
#pragma unroll
            for (int q = 0; q < 11; q++)
                if ((ex[q] >> bit) & 1u) pw[q] = mulm(pw[q], sq);
            if ((top >> (bit + 1)) != 0u) sq = mulm(sq, sq);
        }
        const uint32_t ra = pw[0], rb = pw[1], rc = pw[2];
        uint32_t kres[4], jr[4];
#pragma unroll
        for (int l = 1; l <= 4; l++) {
            kres[l - 1] = a - b - l >= 0 ? pw[2 + l] : 0u;
            jr[l - 1] = a - c - l >= 0 ? pw[6 + l] : 0u;
        }
        // Fermat inverses of rc and the jr (exponent p - 2, per lane), five
        // independent chains in one loop; a zero base has no inverse and is
        // gated (the reference only inverts nonzero powers)
        uint32_t ib[5] = {rc, jr[0], jr[1], jr[2], jr[3]}, iv[5] = {1u, 1u, 1u, 1u, 1u};
        for (uint32_t ee = p - 2u; ee != 0u; ee >>= 1) {
#pragma unroll
            for (int q = 0; q < 5; q++) {
                if (ee & 1u) iv[q] = mulm(iv[q], ib[q]);
                ib[q] = mulm(ib[q], ib[q]);
            }
        }
        const uint32_t ra1 = ra ? ra - 1u : p - 1u;
        uint32_t flags = 0;
        uint32_t un0 = 0, bstep = 0;
        if (rc != 0u) {
            const uint32_t x = mulm(ra1, iv[0]);
            un0 = x ? x - 1u : p - 1u;            // ((ra-1)/rc - 1) mod p
            bstep = mulm(rb, iv[0]);              // rb/rc mod p
            flags |= 1u;
        }
        uint32_t jinv[4];
#pragma unroll
        for (int l = 0; l < 4; l++) jinv[l] = jr[l] ? iv[1 + l] : 0u;
        e[TT_P * TD_SMALL_CAP] = p;
        e[TT_MAGIC * TD_SMALL_CAP] = magic;
        e[TT_UN0 * TD_SMALL_CAP] = un0;
        e[TT_B * TD_SMALL_CAP] = bstep;
        for (int lj = 0; lj < 4; lj++) {
            const uint32_t x = mulm(ra1, jinv[lj]);
            e[(TT_CM + lj) * TD_SMALL_CAP] = x ? x - 1u : p - 1u;
        }
        for (int lk = 0; lk < 4; lk++)
            for (int lj = 0; lj < 4; lj++) {
                e[(TT_E + lk * 4 + lj) * TD_SMALL_CAP] = mulm(kres[lk], jinv[lj]);
                if (kres[lk] != 0u && jinv[lj] != 0u) flags |= 1u << (1 + lk * 4 + lj);
            }
        e[TT_FLAGS * TD_SMALL_CAP] = flags;
        const int f = td_fill_index(p);
        if (f >= 0) {
            // copies of one prime have equal entries, so any writer's index serves
            ctrl[CT_FILL_IDX + f] = i;
            atomicOr(&ctrl[CT_FILL], 1u << f);
        }
    }
}

__device__ __forceinline__ void td_lds_mark(uint32_t *lds, uint32_t bit)
{
    atomicOr(&lds[bit >> 5], 1u << (bit & 31u));
}

// Every mark of one small prime (entry e) in row k: the normal solve, then
// each rev digit group separately (any a - c).
template <int DJ>
__device__ __forceinline__ void td_row_prime(const uint32_t *__restrict__ e, uint32_t k, int lk,
                                             uint32_t rk, uint32_t rowbit, uint32_t J,
                                             uint32_t *lds)
{
    const uint32_t p = e[TT_P * TD_SMALL_CAP], magic = e[TT_MAGIC * TD_SMALL_CAP];
    const uint32_t flags = e[TT_FLAGS * TD_SMALL_CAP];
    if (flags & 1u) {
        const uint32_t u = pf_submod(e[TT_UN0 * TD_SMALL_CAP],
                                     td_mod(k * e[TT_B * TD_SMALL_CAP], p, magic), p);
        for (uint32_t j = u + 1u; j <= J; j += p) td_lds_mark(lds, rowbit + j);
    }
#pragma unroll
    for (int lj = 1; lj <= DJ; lj++) {
        if (!((flags >> (1 + (lk - 1) * 4 + (lj - 1))) & 1u)) continue;
        const uint32_t ev = e[(TT_E + (lk - 1) * 4 + (lj - 1)) * TD_SMALL_CAP];
        const uint32_t u = pf_submod(e[(TT_CM + lj - 1) * TD_SMALL_CAP],
                                     td_mod(rk * ev, p, magic), p);
        const uint32_t lim = td_pow10(lj);
        for (uint32_t r = u + 1u; r < lim; r += p) {
            if (r % 10u == 0u) continue;
            const uint32_t j = td_reverse(r, lj);
            if (j <= J) td_lds_mark(lds, rowbit + j);
        }
    }
}

template <int DJ>
__global__ __launch_bounds__(TD_BLOCK)
void td_rows_kernel(const uint32_t *__restrict__ tbl, const uint32_t *__restrict__ ctrl,
                    uint32_t K, uint32_t J, uint32_t *__restrict__ bits)
{
    extern __shared__ uint32_t lds[];
    const uint32_t k0 = blockIdx.x * TD_ROWS + 1u;
    const uint32_t k_last = min(k0 + TD_ROWS - 1u, K);
    const uint32_t w0 = ((k0 - 1u) * J) >> 5;
    const uint32_t nw = ((k_last * J - 1u) >> 5) - w0 + 1u;
    for (uint32_t w = threadIdx.x; w < nw; w += TD_BLOCK) lds[w] = 0u;
    __syncthreads();

    const uint32_t count = min(ctrl[CT_SMALL_COUNT], TD_SMALL_CAP);
    const uint32_t row = threadIdx.x % TD_ROWS;
    const uint32_t slot = blockIdx.y * (TD_BLOCK / TD_ROWS) + threadIdx.x / TD_ROWS;
    const uint32_t nslots = gridDim.y * (TD_BLOCK / TD_ROWS);
    const uint32_t k = k0 + row;
    if (k <= K) {
        const int lk = td_ndigits(k);
        const uint32_t rk = td_reverse(k, lk);
        // LDS-relative bit of (k, j) is rowbit + j.
        const uint32_t rowbit = (k - 1u) * J - (w0 << 5) - 1u;
        for (uint32_t i = slot; i < count; i += nslots)
            td_row_prime<DJ>(tbl + i, k, lk, rk, rowbit, J, lds);
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < nw; w += TD_BLOCK) {
        const uint32_t v = lds[w];
        if (v) atomicOr(&bits[w0 + w], v);
    }
}

// Work items of the balanced row kernel (one workgroup): per small prime p,
// ceil(ceil(J/p) / TD_CH) normal-solve parts when the solve is active and
// ceil(ceil((10^DJ - 1)/p) / TD_CH) merged-rev parts; p = 2 and 5 (whose
// powers of ten vanish, so digit groups are gated one by one) keep one
// whole-prime item, the fill primes none (the row kernel ORs their class
// masks), and primes with p > J and p >= 10^DJ, which mark at most one j
// per condition and row, one item for both conditions (no mark loop).
// Item = index | kind << 16 | part << 18.
template <int DJ>
__global__ __launch_bounds__(1024)
void td_items_kernel(const uint32_t *__restrict__ tbl, uint32_t *__restrict__ ctrl, uint32_t J,
                     uint32_t *__restrict__ items)
{
    __shared__ uint32_t scan[16];
    const uint32_t count = min(ctrl[CT_SMALL_COUNT], TD_SMALL_CAP);
    const uint32_t per = (count + 1023u) / 1024u;
    const uint32_t i0 = min(threadIdx.x * per, count), i1 = min(i0 + per, count);
    const uint32_t lim = td_pow10(DJ);
    // one item of kind TI_WHOLE or TI_ONE (returned), or nn + nr parts (TI_N)
    auto parts = [&](uint32_t i, uint32_t &nn, uint32_t &nr) -> uint32_t {
        const uint32_t p = tbl[TT_P * TD_SMALL_CAP + i];
        nn = nr = 0;
        if (p == 2u || p == 5u) return TI_WHOLE;
        if (td_fill_index(p) >= 0) return TI_N;                          // word fills
        if (p > J && p >= lim) return TI_ONE;
        const uint32_t flags = tbl[TT_FLAGS * TD_SMALL_CAP + i];
        nn = (flags & 1u) ? ((J + p - 1u) / p + TD_CH - 1u) / TD_CH : 0u;
        nr = ((lim - 1u + p - 1u) / p + TD_CH - 1u) / TD_CH;
        return TI_N;
    };
    uint32_t mine = 0;
    for (uint32_t i = i0; i < i1; i++) {
        uint32_t nn, nr;
        mine += parts(i, nn, nr) != TI_N ? 1u : nn + nr;
    }
    // exclusive offsets: a scan within each wave by lane shuffles, then the
    // 16 wave totals through LDS (one barrier)
    const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
    uint32_t incl = mine;
    for (uint32_t d = 1; d < 64u; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    if (lane == 63u) scan[wid] = incl;
    __syncthreads();
    uint32_t total = 0;
    for (uint32_t w = 0; w < 16u; w++) {
        if (w == wid) incl += total;
        total += scan[w];
    }
    if (threadIdx.x == 0) {
        ctrl[CT_ITEMS] = total;
        ctrl[CT_ITEM_OVF] = total > TD_ITEM_CAP ? 1u : 0u;
    }
    if (total > TD_ITEM_CAP) return;
    uint32_t at = incl - mine;
    for (uint32_t i = i0; i < i1; i++) {
        uint32_t nn, nr;
        const uint32_t kind = parts(i, nn, nr);
        if (kind != TI_N) {
            items[at++] = i | kind << 16;
            continue;
        }
        for (uint32_t q = 0; q < nn; q++) items[at++] = i | (uint32_t)TI_N << 16 | q << 18;
        for (uint32_t q = 0; q < nr; q++) items[at++] = i | (uint32_t)TI_REV << 16 | q << 18;
    }
}

// Class masks of the fill primes for rows of J bits (layout at
// TD_FILL_WORDS).  One lane per mask word.
template <int DJ>
__global__ __launch_bounds__(TD_BLOCK)
void td_fill_table_kernel(uint32_t J, uint32_t *__restrict__ tab)
{
    const uint32_t qw = (J + 31u) >> 5;
    const uint32_t total = 2u * TD_FILL_CLASSES * qw;
    for (uint32_t idx = blockIdx.x * TD_BLOCK + threadIdx.x; idx < total;
         idx += gridDim.x * TD_BLOCK) {
        const uint32_t row = idx / qw, q = idx - row * qw;
        const uint32_t kind = row >= TD_FILL_CLASSES ? 1u : 0u;
        const uint32_t cls = row - kind * TD_FILL_CLASSES;
        int f = 0;
        while (f + 1 < TD_NFILL && c_fill_off[f + 1] <= cls) f++;
        const uint32_t p = c_fill_p[f], r = cls - c_fill_off[f];
        uint32_t w = 0;
        for (uint32_t i = 0; i < 32u; i++) {
            const uint32_t j = q * 32u + i + 1u;
            if (j > J) break;
            uint32_t x = j;
            if (kind) {
                const int lj = td_ndigits(j);
                x = td_reverse(j, lj) * td_pow10(DJ - lj);
            }
            if (x % p == r) w |= 1u << i;
        }
        tab[idx] = w;
    }
}

// Row kernel with merged rev residues (a - c >= DJ): lanes spread over
// (row, work item) instead of (row, prime), so the many marks of the
// smallest primes are shared by many lanes.  rdec is the DJ-digit decode
// table.  Falls back to whole primes if the item list overflowed.  The
// band's items are strided over its gridDim.y workgroups.  The fill primes present in the list (ctrl[CT_FILL]) are marked first, a word
// at a time: per row and fill prime the N condition's hits are the j of one
// class mod p (j = u + 1 + t p) and the rev condition's the j whose R(j) is
// of one class, so the row's words are ORs of the table's class masks,
// shifted to the row's bit offset.
template <int DJ>
__global__ __launch_bounds__(TD_BLOCK)
void td_rows_bal_kernel(const uint32_t *__restrict__ tbl, const uint32_t *__restrict__ ctrl,
                        const uint32_t *__restrict__ items, const uint16_t *__restrict__ rdec,
                        const uint32_t *__restrict__ ftab,
                        uint32_t K, uint32_t J, uint32_t *__restrict__ bits)
{
    extern __shared__ uint32_t lds[];
    constexpr uint32_t NONE = 0xFFFFFFFFu;
    __shared__ uint32_t fmask_at[TD_ROWS][2][TD_NFILL];   // class-mask word offsets, or NONE
    const uint32_t k0 = blockIdx.x * TD_ROWS + 1u;
    const uint32_t k_last = min(k0 + TD_ROWS - 1u, K);
    const uint32_t w0 = ((k0 - 1u) * J) >> 5;
    const uint32_t nw = ((k_last * J - 1u) >> 5) - w0 + 1u;
    for (uint32_t w = threadIdx.x; w < nw; w += TD_BLOCK) lds[w] = 0u;
    // one of the band's gridDim.y workgroups marks the fill primes
    const uint32_t fill = blockIdx.y ? 0u : ctrl[CT_FILL];
    const uint32_t qw = (J + 31u) >> 5;
    if (fill && threadIdx.x < TD_ROWS * TD_NFILL) {
        const uint32_t r = threadIdx.x / TD_NFILL, f = threadIdx.x - r * TD_NFILL;
        const uint32_t kk = k0 + r;
        uint32_t at_n = NONE, at_r = NONE;
        if (kk <= K && ((fill >> f) & 1u)) {
            const uint32_t *e = tbl + ctrl[CT_FILL_IDX + f];
            const uint32_t p = e[TT_P * TD_SMALL_CAP], magic = e[TT_MAGIC * TD_SMALL_CAP];
            const uint32_t flags = e[TT_FLAGS * TD_SMALL_CAP];
            if (flags & 1u) {
                const uint32_t u = pf_submod(e[TT_UN0 * TD_SMALL_CAP],
                                             td_mod(kk * e[TT_B * TD_SMALL_CAP], p, magic), p);
                const uint32_t cls = u + 1u == p ? 0u : u + 1u;
                at_n = (c_fill_off[f] + cls) * qw;
            }
            const int lk = td_ndigits(kk);
            if ((flags >> (1 + (lk - 1) * 4 + (DJ - 1))) & 1u) {
                const uint32_t ev = e[(TT_E + (lk - 1) * 4 + (DJ - 1)) * TD_SMALL_CAP];
                const uint32_t u = pf_submod(e[(TT_CM + DJ - 1) * TD_SMALL_CAP],
                                             td_mod(td_reverse(kk, lk) * ev, p, magic), p);
                const uint32_t cls = u + 1u == p ? 0u : u + 1u;
                at_r = (TD_FILL_CLASSES + c_fill_off[f] + cls) * qw;
            }
        }
        fmask_at[r][0][f] = at_n;
        fmask_at[r][1][f] = at_r;
    }
    __syncthreads();

    if (fill) {
        for (uint32_t t = threadIdx.x; t < TD_ROWS * qw; t += TD_BLOCK) {
            const uint32_t r = t / qw, q = t - r * qw;
            if (k0 + r > K) break;
            uint32_t m = 0;
#pragma unroll
            for (int f = 0; f < TD_NFILL; f++) {
                const uint32_t an = fmask_at[r][0][f], ar = fmask_at[r][1][f];
                if (an != NONE) m |= ftab[an + q];
                if (ar != NONE) m |= ftab[ar + q];
            }
            if (!m) continue;
            // LDS bit of (k0 + r, j = 32 q + 1 + i) is b0 + i; the masks hold no j > J
            const uint32_t b0 = (k0 + r - 1u) * J - (w0 << 5) + (q << 5);
            const uint32_t sh = b0 & 31u, w = b0 >> 5;
            atomicOr(&lds[w], m << sh);
            if (sh) {
                const uint32_t hi = m >> (32u - sh);
                if (hi) atomicOr(&lds[w + 1u], hi);
            }
        }
    }

    const uint32_t row = threadIdx.x % TD_ROWS;
    const uint32_t slot = blockIdx.y * (TD_BLOCK / TD_ROWS) + threadIdx.x / TD_ROWS;
    const uint32_t nslots = gridDim.y * (TD_BLOCK / TD_ROWS);
    const uint32_t k = k0 + row;
    if (k <= K) {
        const int lk = td_ndigits(k);
        const uint32_t rk = td_reverse(k, lk);
        const uint32_t rowbit = (k - 1u) * J - (w0 << 5) - 1u;
        if (ctrl[CT_ITEM_OVF]) {
            const uint32_t count = min(ctrl[CT_SMALL_COUNT], TD_SMALL_CAP);
            for (uint32_t i = slot; i < count; i += nslots)
                td_row_prime<DJ>(tbl + i, k, lk, rk, rowbit, J, lds);
        } else {
            const uint32_t n_items = ctrl[CT_ITEMS];
            const uint32_t lim = td_pow10(DJ);
            const int fbit = 1 + (lk - 1) * 4 + (DJ - 1);
            for (uint32_t it = slot; it < n_items; it += nslots) {
                const uint32_t item = items[it];
                const uint32_t *e = tbl + (item & 0xFFFFu);
                const uint32_t kind = (item >> 16) & 3u, part = item >> 18;
                if (kind == TI_WHOLE) {
                    td_row_prime<DJ>(e, k, lk, rk, rowbit, J, lds);
                    continue;
                }
                const uint32_t p = e[TT_P * TD_SMALL_CAP], magic = e[TT_MAGIC * TD_SMALL_CAP];
                if (kind == TI_ONE) {       // p > J, p >= 10^DJ: at most one mark each
                    const uint32_t flags = e[TT_FLAGS * TD_SMALL_CAP];
                    if (flags & 1u) {
                        const uint32_t u = pf_submod(e[TT_UN0 * TD_SMALL_CAP],
                                                     td_mod(k * e[TT_B * TD_SMALL_CAP], p, magic), p);
                        if (u < J) td_lds_mark(lds, rowbit + u + 1u);
                    }
                    if ((flags >> fbit) & 1u) {
                        const uint32_t ev = e[(TT_E + (lk - 1) * 4 + (DJ - 1)) * TD_SMALL_CAP];
                        const uint32_t u = pf_submod(e[(TT_CM + DJ - 1) * TD_SMALL_CAP],
                                                     td_mod(rk * ev, p, magic), p);
                        if (u + 1u < lim) {
                            const uint32_t j = rdec[u + 1u];
                            if (j <= J) td_lds_mark(lds, rowbit + j);
                        }
                    }
                    continue;
                }
                if (kind == TI_N) {
                    const uint32_t u = pf_submod(e[TT_UN0 * TD_SMALL_CAP],
                                                 td_mod(k * e[TT_B * TD_SMALL_CAP], p, magic), p);
                    uint32_t j = u + 1u + part * TD_CH * p;
                    for (uint32_t t = 0; t < TD_CH && j <= J; t++, j += p)
                        td_lds_mark(lds, rowbit + j);
                } else {
                    const uint32_t flags = e[TT_FLAGS * TD_SMALL_CAP];
                    if (!((flags >> fbit) & 1u)) continue;
                    const uint32_t ev = e[(TT_E + (lk - 1) * 4 + (DJ - 1)) * TD_SMALL_CAP];
                    const uint32_t u = pf_submod(e[(TT_CM + DJ - 1) * TD_SMALL_CAP],
                                                 td_mod(rk * ev, p, magic), p);
                    uint32_t r = u + 1u + part * TD_CH * p;
                    for (uint32_t t = 0; t < TD_CH && r < lim; t++, r += p) {
                        const uint32_t j = rdec[r];
                        if (j <= J) td_lds_mark(lds, rowbit + j);
                    }
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < nw; w += TD_BLOCK) {
        const uint32_t v = lds[w];
        if (v) atomicOr(&bits[w0 + w], v);
    }
}

__device__ __forceinline__ void td_gmark(uint32_t *bits, uint32_t bit)
{
    __hip_atomic_fetch_or(&bits[bit >> 5], 1u << (bit & 31u), __ATOMIC_RELAXED,
                          __HIP_MEMORY_SCOPE_AGENT);
}

// Rare path of the lane kernel: emit every hit of row k.  The lane kernel
// only sees p >= TD_SMALL_LIMIT > 9999 >= max(J, 10^D_j - 1), so each
// residue names at most one j.
//
// Separate groups (MERGED = false): residue l belongs to j digit group l+1;
// its value v is rev(j) - 1 for the j it eliminates, and rev(j) must not end
// in 0 (such a value belongs to no (l+1)-digit j).
// Merged groups (MERGED = true, needs a-c >= DJ): one residue v = R - 1 with
// R = rev(j) 10^(DJ - lj), i.e. rev(j) padded with zeros to DJ digits, which
// names (lj, rev(j)) uniquely; rdec[R] holds that j (td_rdec_kernel).
static_assert(TD_SMALL_LIMIT > 9999u, "lane kernel assumes one j per residue");

// Lanes with p >= TD_FIX_MIN track fixed-point images of their residues
// (1 op per residue and k, candidates recomputed exactly).  Smaller primes
// have candidates at more k (a wave of 64 lanes enters the candidate path
// with probability ~64 x 14 095 / p per k), where exact residues (3 ops per
// residue and k, hits read directly) cost less.  Measured per triple at
// K = J = 4096: 4.46 ms with the switch at 2^20, 4.30 at 2^22, 4.23 at
// 2^23, 4.20 at 2^24; 5.17 with exact residues everywhere.
constexpr uint32_t TD_FIX_MIN = 1u << 24;

template <int DJ, bool MERGED, int NR>
__device__ __forceinline__ void td_hits(uint32_t k, uint32_t un, uint32_t thrn,
                                        const uint32_t (&v)[NR], const uint32_t (&thr)[NR],
                                        uint32_t J, const uint16_t *__restrict__ rdec,
                                        uint32_t *bits)
{
    const uint32_t rowbit = (k - 1u) * J - 1u;      // bit of (k, j) = rowbit + j
    if (un < thrn) td_gmark(bits, rowbit + un + 1u);
#pragma unroll
    for (int l = 0; l < NR; l++) {
        if (v[l] < thr[l]) {
            const uint32_t r = v[l] + 1u;
            uint32_t j;
            if (MERGED) {
                j = td_rdec_arith(r, DJ);    // = rdec[r], without the load's latency
            } else {
                j = (r % 10u == 0u) ? 0xFFFFFFFFu : td_reverse(r, l + 1);
            }
            if (j <= J) td_gmark(bits, rowbit + j);
        }
    }
}

// Fixed-point image of a residue x mod p (x < p): round(x 2^32 / p), with
// fp = 2^32 / p in double precision (relative error 2^-52, far below one
// unit).  The image of (x - s) mod p is the image of x minus the image of s
// modulo 2^32, up to one rounding error per subtraction, so a residue is
// advanced with one subtraction (the wrap mod 2^32 is the wrap mod p) and
// tested with one compare against its window widened by the error
// accumulated so far; the rare candidates are recomputed exactly.
__device__ __forceinline__ uint32_t td_fix(uint32_t x, double fp)
{
    return (uint32_t)__double2ull_rn((double)x * fp);
}

// Upper end of the candidate window of residues v < thr, images shifted by
// eoff (the error bound): true hits have images in [0, thr fp + 2 eoff).
__device__ __forceinline__ uint32_t td_fix_window(uint32_t thr, double fp, uint32_t eoff)
{
    return thr ? (uint32_t)ceil((double)thr * fp) + 2u * eoff : 0u;
}

// Candidate of the fixed-point test: the exact residues of row k, then the
// marks of td_hits.  un(k) = un0 - k bstep, v_l(k) = cm_l - rev(k) E_l
// (mod p), rev(k) with lk digits; bstepM and eM_l in Montgomery form.
template <int DJ, bool MERGED, int NR>
__device__ __forceinline__ void td_hits_exact(uint32_t k, int lk, uint32_t un0, uint32_t bstepM,
                                              const uint32_t (&cm)[NR], const uint32_t (&eM)[NR],
                                              const uint32_t (&thr)[NR], PfMont m,
                                              uint32_t J, const uint16_t *__restrict__ rdec,
                                              uint32_t *bits)
{
    const uint32_t p = m.p;
    const uint32_t un = pf_submod(un0, pf_mont_mul(bstepM, k, m), p);
    const uint32_t rk = td_reverse(k, lk);
    uint32_t v[NR];
#pragma unroll
    for (int l = 0; l < NR; l++) v[l] = pf_submod(cm[l], pf_mont_mul(eM[l], rk, m), p);
    td_hits<DJ, MERGED, NR>(k, un, J, v, thr, J, rdec, bits);
}

// True when some lane of the wave has h set: a wave-uniform branch (one
// scalar test), so the loop does not save and restore the exec mask per k.
__device__ __forceinline__ bool td_any(bool h) { return __ballot(h) != 0ull; }

// rdec tables for D = 1..4 at offsets 0, 10, 110, 1110: rdec_D[R] = the j
// whose rev(j) padded with zeros to D digits is R (0 for R = 0).
constexpr uint32_t TD_RDEC_SIZE = 11110;

__device__ __forceinline__ uint32_t td_rdec_offset(int d)
{
    return d <= 1 ? 0u : d == 2 ? 10u : d == 3 ? 110u : 1110u;
}

__global__ void td_rdec_kernel(uint16_t *rdec)
{
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= TD_RDEC_SIZE) return;
    const int d = i < 10u ? 1 : i < 110u ? 2 : i < 1110u ? 3 : 4;
    rdec[i] = (uint16_t)td_rdec_value(i - td_rdec_offset(d), d);
}

template <int DJ, bool MERGED>
__global__ __launch_bounds__(TD_BLOCK)
void td_large_kernel(const uint32_t *__restrict__ primes, uint32_t n,
                     long long a, long long b, long long c,
                     uint32_t K, uint32_t J, const uint16_t *__restrict__ rdec,
                     uint32_t *__restrict__ bits, uint32_t pmax)
{
    constexpr int NR = MERGED ? 1 : DJ;     // rev residues tracked per k
    const uint32_t i = blockIdx.x * TD_BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = primes[i];
    if (p < TD_SMALL_LIMIT || p >= pmax) return;

    // ---- per-prime setup (Montgomery, R = 2^32) ----
    const PfMont m = pf_mont_init(p);
    const uint32_t ten = pf_mont_in(10u, m);
    // 10^{-1}: 10 x = 1 + t p with t p == 9 (mod 10), t fixed by p mod 10.
    const uint32_t pm = p % 10u;
    const uint32_t t = pm == 1u ? 9u : pm == 3u ? 3u : pm == 7u ? 7u : 1u;
    const uint32_t tenInv = pf_mont_in((uint32_t)((1ull + (uint64_t)t * p) / 10u), m);

    const uint32_t raM = pf_mont_pow(ten, (uint64_t)a, m);
    const uint32_t rbM = pf_mont_pow(ten, (uint64_t)b, m);
    const uint32_t icS = pf_mont_out(pf_mont_pow(tenInv, (uint64_t)c, m), m);   // 10^-c
    const uint32_t ra1M = pf_submod(raM, m.one, p);                              // ra - 1
    const uint32_t bstep = pf_mont_mul(rbM, icS, m);                             // rb / rc
    const uint32_t un0 = pf_submod(pf_mont_mul(ra1M, icS, m), 1u, p);            // u at k = 0
    // Rev residue l is (ra - 1 - rev(k) kres) / X_l - 1 with
    //   separate: X_l = 10^(a-c-(l+1)), hit range [0, 10^(l+1) - 1);
    //   merged:   X_0 = 10^(a-c-DJ),    hit range [0, 10^DJ - 1).
    uint32_t jinvM[NR], cm[NR];
    bool jok[NR];
    {
        const long long e1 = MERGED ? a - c - DJ : a - c - 1;
        uint32_t z = e1 >= 0 ? pf_mont_pow(tenInv, (uint64_t)e1, m) : 0u;
#pragma unroll
        for (int l = 0; l < NR; l++) {
            jok[l] = MERGED ? e1 >= 0 : (a - c - (l + 1)) >= 0;
            jinvM[l] = z;
            cm[l] = pf_submod(pf_mont_mul(ra1M, pf_mont_out(z, m), m), 1u, p);
            z = pf_mont_mul(z, ten, m);
        }
    }
    // k digit groups: kres = 10^(a-b-lk), advanced by 10^{-1} per group.
    const long long eb1 = a - b - 1;
    uint32_t kresM = eb1 >= 0 ? pf_mont_pow(ten, (uint64_t)eb1, m) : 0u;

    if (p < TD_FIX_MIN) {
        // exact residues: 3 ops per residue and k, the hit path has them at hand
        uint32_t un = un0;
        const uint32_t thrn = J;
        const int DK = (K >= 1000u) ? 4 : (K >= 100u) ? 3 : (K >= 10u) ? 2 : 1;
        for (int lk = 1; lk <= DK; lk++) {
            const uint32_t klo = td_pow10(lk - 1);
            const uint32_t khi = min(K, td_pow10(lk) - 1u);
            const bool kok = (a - b - lk) >= 0;
            // Steps of rev(k) inside a row of ten (units digit of k -> top digit
            // of rev(k)) and between rows (q -> q+1 with t9 trailing nines).
            const uint32_t s0w = td_pow10(lk - 1);
            uint32_t thr[NR], s0[NR], w[NR], tq0[NR], tq1[NR], tq2[NR];
    #pragma unroll
            for (int l = 0; l < NR; l++) {
                const uint32_t eM = pf_mont_mul(kresM, jinvM[l], m);      // E = kres / X_l
                thr[l] = (kok && jok[l]) ? td_pow10(MERGED ? DJ : l + 1) - 1u : 0u;
                s0[l] = pf_mont_mul(eM, s0w, m);
                const uint32_t eS = pf_mont_out(eM, m);
                w[l] = lk == 1 ? cm[l] : pf_submod(cm[l], eS, p);         // rev(10^(lk-1)) = 1
                // delta_t = 10^(lk-2-t) - 9 * sum_{i<t} 10^(lk-2-i), reduced mod p.
                int d0 = lk >= 2 ? (int)td_pow10(lk - 2) : 0;
                int d1 = lk >= 3 ? (int)td_pow10(lk - 3) - 9 * (int)td_pow10(lk - 2) : 0;
                int d2 = lk >= 4 ? (int)td_pow10(lk - 4) - 9 * ((int)td_pow10(lk - 2) + (int)td_pow10(lk - 3)) : 0;
                tq0[l] = pf_mont_mul(eM, d0 >= 0 ? (uint32_t)d0 : p - (uint32_t)(-d0), m);
                tq1[l] = pf_mont_mul(eM, d1 >= 0 ? (uint32_t)d1 : p - (uint32_t)(-d1), m);
                tq2[l] = pf_mont_mul(eM, d2 >= 0 ? (uint32_t)d2 : p - (uint32_t)(-d2), m);
            }

            const uint32_t qlo = klo / 10u, qhi = khi / 10u;
            for (uint32_t q = qlo; q <= qhi; q++) {
                const uint32_t kb = q * 10u;
                const uint32_t dlo = kb < klo ? klo - kb : 0u;
                const uint32_t dhi = min(9u, khi - kb);
                uint32_t v[NR];
    #pragma unroll
                for (int l = 0; l < NR; l++) v[l] = w[l];
                if (dlo == 0u && dhi == 9u) {
    #pragma unroll
                    for (uint32_t d = 0; d < 10u; d++) {
                        un = pf_submod(un, bstep, p);
                        bool h = un < thrn;
    #pragma unroll
                        for (int l = 0; l < NR; l++) h |= v[l] < thr[l];
                        if (__builtin_expect(td_any(h), 0))
                            if (h) td_hits<DJ, MERGED, NR>(kb + d, un, thrn, v, thr, J, rdec, bits);
    #pragma unroll
                        for (int l = 0; l < NR; l++) v[l] = pf_submod(v[l], s0[l], p);
                    }
                } else {
                    for (uint32_t d = 0; d < dlo; d++) {
    #pragma unroll
                        for (int l = 0; l < NR; l++) v[l] = pf_submod(v[l], s0[l], p);
                    }
                    for (uint32_t d = dlo; d <= dhi; d++) {
                        un = pf_submod(un, bstep, p);
                        bool h = un < thrn;
    #pragma unroll
                        for (int l = 0; l < NR; l++) h |= v[l] < thr[l];
                        if (h) td_hits<DJ, MERGED, NR>(kb + d, un, thrn, v, thr, J, rdec, bits);
    #pragma unroll
                        for (int l = 0; l < NR; l++) v[l] = pf_submod(v[l], s0[l], p);
                    }
                }
                if (q < qhi) {
                    uint32_t t9 = 0, qq = q;
                    while (qq % 10u == 9u) { t9++; qq /= 10u; }
    #pragma unroll
                    for (int l = 0; l < NR; l++)
                        w[l] = pf_submod(w[l], t9 == 0 ? tq0[l] : t9 == 1 ? tq1[l] : tq2[l], p);
                }
            }
            kresM = pf_mont_mul(kresM, tenInv, m);
        }
        return;
    }
    // fixed-point images: 1 op per residue and k, candidates recomputed exactly
    // Fixed-point images (td_fix).  Every image below is derived from an
    // exact residue once per prime (un) or once per digit count of k (the
    // rev residues) and then advanced at most K + 1 times, half a unit of
    // error each, so eoff = 2K + 32 bounds the error.
    const double fp = 4294967296.0 / (double)p;
    const uint32_t eoff = 2u * K + 32u;
    const uint32_t bF = td_fix(bstep, fp);
    const uint32_t tU = td_fix_window(J, fp, eoff);
    const uint32_t bstepM = pf_mont_in(bstep, m);
    uint32_t uF = td_fix(un0, fp) + eoff;
    const int DK = (K >= 1000u) ? 4 : (K >= 100u) ? 3 : (K >= 10u) ? 2 : 1;
    for (int lk = 1; lk <= DK; lk++) {
        const uint32_t klo = td_pow10(lk - 1);
        const uint32_t khi = min(K, td_pow10(lk) - 1u);
        const bool kok = (a - b - lk) >= 0;
        const uint32_t s0w = td_pow10(lk - 1);
        // exact per class (for the candidates' recheck): thr, E_l; images of
        // the row start w, the in-row step s0 and the row-to-row steps tq
        uint32_t thr[NR], eMl[NR], tV[NR], sF[NR], wF[NR], q0F[NR], q1F[NR], q2F[NR];
#pragma unroll
        for (int l = 0; l < NR; l++) {
            const uint32_t eM = pf_mont_mul(kresM, jinvM[l], m);      // E = kres / X_l
            eMl[l] = eM;
            thr[l] = (kok && jok[l]) ? td_pow10(MERGED ? DJ : l + 1) - 1u : 0u;
            tV[l] = td_fix_window(thr[l], fp, eoff);
            sF[l] = td_fix(pf_mont_mul(eM, s0w, m), fp);
            const uint32_t eS = pf_mont_out(eM, m);
            wF[l] = td_fix(lk == 1 ? cm[l] : pf_submod(cm[l], eS, p), fp) + eoff;   // rev(10^(lk-1)) = 1
            // delta_t = 10^(lk-2-t) - 9 * sum_{i<t} 10^(lk-2-i), reduced mod p.
            int d0 = lk >= 2 ? (int)td_pow10(lk - 2) : 0;
            int d1 = lk >= 3 ? (int)td_pow10(lk - 3) - 9 * (int)td_pow10(lk - 2) : 0;
            int d2 = lk >= 4 ? (int)td_pow10(lk - 4) - 9 * ((int)td_pow10(lk - 2) + (int)td_pow10(lk - 3)) : 0;
            q0F[l] = td_fix(pf_mont_mul(eM, d0 >= 0 ? (uint32_t)d0 : p - (uint32_t)(-d0), m), fp);
            q1F[l] = td_fix(pf_mont_mul(eM, d1 >= 0 ? (uint32_t)d1 : p - (uint32_t)(-d1), m), fp);
            q2F[l] = td_fix(pf_mont_mul(eM, d2 >= 0 ? (uint32_t)d2 : p - (uint32_t)(-d2), m), fp);
        }

        const uint32_t qlo = klo / 10u, qhi = khi / 10u;
        for (uint32_t q = qlo; q <= qhi; q++) {
            const uint32_t kb = q * 10u;
            const uint32_t dlo = kb < klo ? klo - kb : 0u;
            const uint32_t dhi = min(9u, khi - kb);
            uint32_t vF[NR];
#pragma unroll
            for (int l = 0; l < NR; l++) vF[l] = wF[l];
            if (dlo == 0u && dhi == 9u) {
#pragma unroll
                for (uint32_t d = 0; d < 10u; d++) {
                    uF -= bF;
                    bool h = uF < tU;
#pragma unroll
                    for (int l = 0; l < NR; l++) h |= vF[l] < tV[l];
                    if (__builtin_expect(td_any(h), 0))
                        if (h) td_hits_exact<DJ, MERGED, NR>(kb + d, lk, un0, bstepM, cm, eMl, thr, m, J, rdec, bits);
#pragma unroll
                    for (int l = 0; l < NR; l++) vF[l] -= sF[l];
                }
            } else {
                for (uint32_t d = 0; d < dlo; d++) {
#pragma unroll
                    for (int l = 0; l < NR; l++) vF[l] -= sF[l];
                }
                for (uint32_t d = dlo; d <= dhi; d++) {
                    uF -= bF;
                    bool h = uF < tU;
#pragma unroll
                    for (int l = 0; l < NR; l++) h |= vF[l] < tV[l];
                    if (h) td_hits_exact<DJ, MERGED, NR>(kb + d, lk, un0, bstepM, cm, eMl, thr, m, J, rdec, bits);
#pragma unroll
                    for (int l = 0; l < NR; l++) vF[l] -= sF[l];
                }
            }
            if (q < qhi) {
                uint32_t t9 = 0, qq = q;
                while (qq % 10u == 9u) { t9++; qq /= 10u; }
#pragma unroll
                for (int l = 0; l < NR; l++) wF[l] -= t9 == 0 ? q0F[l] : t9 == 1 ? q1F[l] : q2F[l];
            }
        }
        kresM = pf_mont_mul(kresM, tenInv, m);
    }
}

// Mid-range primes (from 2^16 up to the lattice path, merged j digit
// groups), exact residues: the k loop of td_large_kernel with each prime's
// rows split over TD_MID_SPLIT lanes (q ranges of k / 10), so that the
// ~10^5 primes of the range fill the machine (one lane per prime left most
// SIMDs idle).  The lanes of one prime repeat the setup (they run side by
// side in one wave, so it costs no extra time) and start their residues at
// their own first row: u = un0 - k0 rb/rc and the rev residue
// cm - rev(10 q0) E (one Montgomery product each).  Grid-stride over the
// compacted list td_split_kernel wrote.
#ifndef TD_MID_SPLIT_N
#define TD_MID_SPLIT_N 8
#endif
constexpr int TD_MID_SPLIT = TD_MID_SPLIT_N;

template <int DJ>
__global__ __launch_bounds__(TD_BLOCK)
void td_mid_kernel(const uint32_t *__restrict__ mid, const uint32_t *__restrict__ ctrl,
                   long long a, long long b, long long c,
                   uint32_t K, uint32_t J, const uint16_t *__restrict__ rdec,
                   uint32_t *__restrict__ bits)
{
    const uint32_t count = min(ctrl[CT_MID_COUNT], TD_MID_CAP);
    const uint32_t Qtot = K / 10u + 1u;           // q = k / 10 runs over [0, Qtot)
    const int DK = (K >= 1000u) ? 4 : (K >= 100u) ? 3 : (K >= 10u) ? 2 : 1;
    const uint32_t thr = td_pow10(DJ) - 1u;
    for (uint32_t g = blockIdx.x * TD_BLOCK + threadIdx.x; g < count * TD_MID_SPLIT;
         g += gridDim.x * TD_BLOCK) {
        const uint32_t p = mid[g / TD_MID_SPLIT];
        const uint32_t part = g % TD_MID_SPLIT;
        const uint32_t qa = part * Qtot / TD_MID_SPLIT, qb = (part + 1u) * Qtot / TD_MID_SPLIT;
        if (qa >= qb) continue;

        // ---- per-prime setup (Montgomery, R = 2^32) ----
        const PfMont m = pf_mont_init(p);
        const uint32_t ten = pf_mont_in(10u, m);
        const uint32_t pm = p % 10u;
        const uint32_t t = pm == 1u ? 9u : pm == 3u ? 3u : pm == 7u ? 7u : 1u;
        const uint32_t tenInv = pf_mont_in((uint32_t)((1ull + (uint64_t)t * p) / 10u), m);
        const long long eb1 = a - b - 1;
        uint32_t pw[3], nw[2];
        {
            const uint64_t pe[3] = {(uint64_t)a, (uint64_t)b, (uint64_t)(eb1 >= 0 ? eb1 : 0)};
            const uint64_t ne[2] = {(uint64_t)c, (uint64_t)(a - c - DJ)};
            pf_mont_pow_multi<3>(ten, pe, pw, m);
            pf_mont_pow_multi<2>(tenInv, ne, nw, m);
        }
        const uint32_t icS = pf_mont_out(nw[0], m);                                 // 10^-c
        const uint32_t ra1M = pf_submod(pw[0], m.one, p);                           // ra - 1
        const uint32_t bstep = pf_mont_mul(pw[1], icS, m);                          // rb / rc
        const uint32_t bstepM = pf_mont_in(bstep, m);
        const uint32_t un0 = pf_submod(pf_mont_mul(ra1M, icS, m), 1u, p);           // u at k = 0
        const uint32_t jinvM = nw[1];                                               // 10^-(a-c-DJ)
        const uint32_t cm = pf_submod(pf_mont_mul(ra1M, pf_mont_out(jinvM, m), m), 1u, p);
        uint32_t kresM = pw[2];                                                     // 10^(a-b-lk)
        const uint32_t thrn = J;
        for (int lk = 1; lk <= DK; lk++) {
            const uint32_t klo = td_pow10(lk - 1);
            const uint32_t khi = min(K, td_pow10(lk) - 1u);
            const uint32_t qlo = klo / 10u, qhi = khi / 10u;
            const uint32_t q0 = max(qlo, qa), q1 = min(qhi, qb - 1u);
            if (q0 <= q1) {
                const bool kok = (a - b - lk) >= 0 && eb1 >= 0;
                const uint32_t s0w = td_pow10(lk - 1);
                const uint32_t eM = pf_mont_mul(kresM, jinvM, m);          // E = kres / X_0
                const uint32_t th = kok ? thr : 0u;
                const uint32_t s0 = pf_mont_mul(eM, s0w, m);
                // rev residue at the lane's first row start k = 10 q0 (the
                // class's first k, rev = 1, when the lane starts the class)
                uint32_t w = q0 == qlo ? (lk == 1 ? cm : pf_submod(cm, pf_mont_out(eM, m), p))
                                       : pf_submod(cm, pf_mont_mul(eM, td_reverse(10u * q0, lk), m), p);
                // N residue before the lane's first k of the class
                const uint32_t k0 = max(klo, 10u * q0);
                uint32_t un = pf_submod(un0, pf_mont_mul(bstepM, k0 - 1u, m), p);
                int d0 = lk >= 2 ? (int)td_pow10(lk - 2) : 0;
                int d1 = lk >= 3 ? (int)td_pow10(lk - 3) - 9 * (int)td_pow10(lk - 2) : 0;
                int d2 = lk >= 4 ? (int)td_pow10(lk - 4) - 9 * ((int)td_pow10(lk - 2) + (int)td_pow10(lk - 3)) : 0;
                const uint32_t tq0 = pf_mont_mul(eM, d0 >= 0 ? (uint32_t)d0 : p - (uint32_t)(-d0), m);
                const uint32_t tq1 = pf_mont_mul(eM, d1 >= 0 ? (uint32_t)d1 : p - (uint32_t)(-d1), m);
                const uint32_t tq2 = pf_mont_mul(eM, d2 >= 0 ? (uint32_t)d2 : p - (uint32_t)(-d2), m);
                for (uint32_t q = q0; q <= q1; q++) {
                    const uint32_t kb = q * 10u;
                    const uint32_t dlo = kb < klo ? klo - kb : 0u;
                    const uint32_t dhi = min(9u, khi - kb);
                    uint32_t v[1] = {w};
                    const uint32_t thv[1] = {th};
                    for (uint32_t d = 0; d < dlo; d++) v[0] = pf_submod(v[0], s0, p);
                    for (uint32_t d = dlo; d <= dhi; d++) {
                        un = pf_submod(un, bstep, p);
                        const bool h = un < thrn || v[0] < th;
                        if (__builtin_expect(td_any(h), 0))
                            if (h) td_hits<DJ, true, 1>(kb + d, un, thrn, v, thv, J, rdec, bits);
                        v[0] = pf_submod(v[0], s0, p);
                    }
                    if (q < q1) {
                        uint32_t t9 = 0, qq = q;
                        while (qq % 10u == 9u) { t9++; qq /= 10u; }
                        w = pf_submod(w, t9 == 0 ? tq0 : t9 == 1 ? tq1 : tq2, p);
                    }
                }
            }
            kresM = pf_mont_mul(kresM, tenInv, m);
        }
    }
}

// Lattice kernel: primes >= TD_LAT_MIN (merged j digit groups), hits
// enumerated directly (td_lattice.h) instead of the K-step loop of
// td_large_kernel: one lane per prime, its four condition searches in turn.
// (A per-wave queue that hands exhausted lanes the next search balanced the
// lanes but cost more in bookkeeping than it saved: 2.29 against 1.92 ms
// per 4096 x 4096 triple over the primes below 10^8.)
#ifndef TD_LAT_MIN_LOG2
#define TD_LAT_MIN_LOG2 17
#endif
constexpr uint32_t TD_LAT_MIN = 1u << TD_LAT_MIN_LOG2;
static_assert(TD_LAT_MIN >= TD_SMALL_LIMIT, "the lattice path needs p > 10^4 >= J");
static_assert(TD_LAT_MIN <= (1u << 24), "every prime of [2^16, TD_LAT_MIN) fits the mid list");

struct TdDevMark {
    uint32_t *bits;
    __device__ __forceinline__ void operator()(uint32_t bit) const { td_gmark(bits, bit); }
};

template <int DJ>
__global__ __launch_bounds__(TD_BLOCK)
void td_lattice_kernel(const uint32_t *__restrict__ primes, uint32_t n,
                       long long a, long long b, long long c,
                       uint32_t K, uint32_t J, uint32_t wtop, uint32_t *__restrict__ bits,
                       uint32_t pmin)
{
    const uint32_t i = blockIdx.x * TD_BLOCK + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = primes[i];
    if (p < pmin || p >= TD_PMAX) return;
    TdDevMark mark{bits};
    td_lattice_prime<DJ>(p, a, b, c, K, J, wtop, mark);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

constexpr int TD_MAX_DEV = 64;
constexpr uint32_t TD_RDEC_OFF[5] = {0u, 0u, 10u, 110u, 1110u};

struct TdScratch {
    bool ready = false;          // every field below allocated and initialised
    uint32_t *small = nullptr;   // [TD_SMALL_CAP]
    uint32_t *tbl = nullptr;     // [TD_SMALL_CAP * TD_TBL]
    uint32_t *ctrl = nullptr;    // [CT_WORDS]
    uint16_t *rdec = nullptr;    // [TD_RDEC_SIZE]
    uint32_t *items = nullptr;   // [TD_ITEM_CAP] row-kernel work items
    uint32_t *mid = nullptr;     // [TD_MID_CAP] compacted mid-range primes
    uint32_t *fill = nullptr;    // [TD_FILL_WORDS] class masks of the fill primes
    uint32_t fill_J = 0;         // the J the class masks were built for (0: none)
    uint32_t *fill_key = nullptr; // where that J is kept across calls (this struct's
                                  // own field, or the allocation-free state's)
    hipStream_t aux = nullptr;   // row kernel, concurrent with the lane kernel
    hipEvent_t fork = nullptr, join = nullptr;
};

TdScratch g_scratch[TD_MAX_DEV];

void td_scratch_release(TdScratch &s)
{
    if (s.small) (void)hipFree(s.small);
    if (s.tbl) (void)hipFree(s.tbl);
    if (s.ctrl) (void)hipFree(s.ctrl);
    if (s.rdec) (void)hipFree(s.rdec);
    if (s.items) (void)hipFree(s.items);
    if (s.mid) (void)hipFree(s.mid);
    if (s.fill) (void)hipFree(s.fill);
    if (s.aux) (void)hipStreamDestroy(s.aux);
    if (s.fork) (void)hipEventDestroy(s.fork);
    if (s.join) (void)hipEventDestroy(s.join);
    s = TdScratch{};
}

// Per-device scratch, set up on first use.  A failed set-up releases what it
// allocated, so the next call tries again from scratch.
int td_scratch(TdScratch **out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= TD_MAX_DEV) return -1;
    TdScratch &s = g_scratch[dev];
    if (!s.ready) {
        bool ok = hipMalloc(&s.small, TD_SMALL_CAP * sizeof(uint32_t)) == hipSuccess &&
                  hipMalloc(&s.tbl, (size_t)TD_SMALL_CAP * TD_TBL * sizeof(uint32_t)) == hipSuccess &&
                  hipMalloc(&s.ctrl, CT_WORDS * sizeof(uint32_t)) == hipSuccess &&
                  hipMemset(s.ctrl, 0, CT_WORDS * sizeof(uint32_t)) == hipSuccess &&
                  hipMalloc(&s.rdec, TD_RDEC_SIZE * sizeof(uint16_t)) == hipSuccess &&
                  hipMalloc(&s.items, TD_ITEM_CAP * sizeof(uint32_t)) == hipSuccess &&
                  hipMalloc(&s.mid, TD_MID_CAP * sizeof(uint32_t)) == hipSuccess &&
                  hipMalloc(&s.fill, TD_FILL_WORDS * sizeof(uint32_t)) == hipSuccess;
        if (ok) {
            td_rdec_kernel<<<(TD_RDEC_SIZE + 255u) / 256u, 256>>>(s.rdec);
            ok = hipGetLastError() == hipSuccess &&
                 hipStreamCreateWithFlags(&s.aux, hipStreamNonBlocking) == hipSuccess &&
                 hipEventCreateWithFlags(&s.fork, hipEventDisableTiming) == hipSuccess &&
                 hipEventCreateWithFlags(&s.join, hipEventDisableTiming) == hipSuccess &&
                 hipDeviceSynchronize() == hipSuccess;
        }
        if (!ok) {
            td_scratch_release(s);
            return -1;
        }
        s.ready = true;
        s.fill_key = &s.fill_J;
    }
    *out = &s;
    return 0;
}

// Workgroups per row band (gridDim.y of the row kernels): they share the
// band's work items and OR their LDS copies of the band into the bitmap.
// A lane's items form a serial chain of dependent loads, so few bands leave
// the chip idle behind it: with one workgroup each the kernel took 131 us at
// 256 x 256 (64 bands) and 180 at 1500 x 777 (375 bands), against 17 and 132
// here; 1024 bands (4096 x 4096) gain 6% from a second one and lose from a
// fourth.  Above 16 the clearing and the merging of the band cost what the
// shorter chains give.
uint32_t td_row_split(uint32_t bands)
{
    return std::max(1u, std::min(16u, 2048u / bands));
}

template <int DJ>
void td_launch_rest(const uint32_t *d_primes, uint32_t n, long long a, long long b,
                    long long c, uint32_t K, uint32_t J, uint32_t *d_bits,
                    const TdScratch &s, hipStream_t st, hipEvent_t ev0, hipEvent_t ev1)
{
    const dim3 row_groups((K + TD_ROWS - 1u) / TD_ROWS,
                          td_row_split((K + TD_ROWS - 1u) / TD_ROWS));
    const size_t lds = ((size_t)TD_ROWS * J / 32u + 2u) * sizeof(uint32_t);
    // The row kernel and the mid-range k loop (both latency-bound: few waves,
    // long dependent chains, frequent hit paths) run in turn on the
    // auxiliary stream beside the lattice or k-loop kernel of the large
    // primes (VALU-bound); all of them only OR into the bitmap.  The join
    // before returning keeps the shared scratch (table, items, mid list)
    // from being overwritten by the next call while they still read it.
    // Without an auxiliary stream (the allocation-free launch) every kernel
    // runs in order on st.
    // (The small primes' setup and work items stay on st, ahead of the fork:
    // queued behind the fork they start only when the large primes' kernel
    // frees compute units, and the row kernel then ends after it: 16.7
    // against 14.9 ms per 8 triples of 4096 x 4096.)
    const hipStream_t rs = s.aux ? s.aux : st;
    if (a - c >= DJ) {
        td_items_kernel<DJ><<<1, 1024, 0, st>>>(s.tbl, s.ctrl, J, s.items);
        // the class masks depend on J alone: built once per device and J
        // (calls on one device are ordered, as they share the scratch)
        if (!s.fill_key || *s.fill_key != J) {
            const uint32_t fw = 2u * TD_FILL_CLASSES * ((J + 31u) >> 5);
            td_fill_table_kernel<DJ><<<(fw + TD_BLOCK - 1u) / TD_BLOCK, TD_BLOCK, 0, st>>>(J, s.fill);
            if (s.fill_key) *s.fill_key = J;
        }
    }
    if (s.aux) {
        (void)hipEventRecord(s.fork, st);
        (void)hipStreamWaitEvent(s.aux, s.fork, 0);
    }
    if (a - c >= DJ)
        td_rows_bal_kernel<DJ><<<row_groups, TD_BLOCK, lds, rs>>>(
            s.tbl, s.ctrl, s.items, s.rdec + TD_RDEC_OFF[DJ], s.fill, K, J, d_bits);
    else
        td_rows_kernel<DJ><<<row_groups, TD_BLOCK, lds, rs>>>(s.tbl, s.ctrl, K, J, d_bits);
    // One merged rev residue per k needs every j digit group's exponent
    // a-c-lj >= 0; otherwise track the groups separately.
    // primes >= TD_LAT_MIN enumerate their hits directly when the j digit
    // groups merge, those from 2^16 below take the split k loop; for
    // separate groups, every prime from 2^16 takes the K-step lane kernel.
    if (n && a - c >= DJ) {
        const uint32_t mid_blocks = std::min<uint64_t>(
            2048u, ((uint64_t)n * TD_MID_SPLIT + TD_BLOCK - 1u) / TD_BLOCK);
        td_mid_kernel<DJ><<<mid_blocks, TD_BLOCK, 0, rs>>>(
            s.mid, s.ctrl, a, b, c, K, J, s.rdec + TD_RDEC_OFF[DJ], d_bits);
    }
    if (s.aux) (void)hipEventRecord(s.join, s.aux);
    if (ev0) (void)hipEventRecord(ev0, st);
    if (n && a - c >= DJ) {
        td_lattice_kernel<DJ><<<(n + TD_BLOCK - 1u) / TD_BLOCK, TD_BLOCK, 0, st>>>(
            d_primes, n, a, b, c, K, J, td_top_window(K), d_bits, TD_LAT_MIN);
    } else if (n) {
        td_large_kernel<DJ, false><<<(n + TD_BLOCK - 1u) / TD_BLOCK, TD_BLOCK, 0, st>>>(
            d_primes, n, a, b, c, K, J, s.rdec + TD_RDEC_OFF[DJ], d_bits, TD_PMAX);
    }
    if (ev1) (void)hipEventRecord(ev1, st);
    if (s.aux) (void)hipStreamWaitEvent(st, s.join, 0);
}

// ---- allocation-free launch (trial_div_launch_kj_noalloc) ----
//
// The same kernels with their scratch (small-prime list, setup table,
// control words, rev(j) decode table, row-kernel items) in one file-scope
// device array instead of hipMalloc'd buffers, and every kernel on the
// caller's stream.  Each device holds its own copy of the array until the
// process ends; its device address is looked up once per device with
// hipGetSymbolAddress (the array's name is not a device address in host
// code).  The control words are cleared by td_reset_kernel / td_items_kernel
// on every call; the error latch is read and cleared by
// trial_div_check_error().
constexpr size_t TD_NA_SMALL = 0;
constexpr size_t TD_NA_TBL   = TD_NA_SMALL + TD_SMALL_CAP;
constexpr size_t TD_NA_CTRL  = TD_NA_TBL + (size_t)TD_SMALL_CAP * TD_TBL;
constexpr size_t TD_NA_RDEC  = TD_NA_CTRL + 64;                      // 256-byte aligned
constexpr size_t TD_NA_ITEMS = TD_NA_RDEC + ((TD_RDEC_SIZE * sizeof(uint16_t) + 255u) / 256u) * 64u;
constexpr size_t TD_NA_MID   = TD_NA_ITEMS + TD_ITEM_CAP;
constexpr size_t TD_NA_FILL  = TD_NA_MID + TD_MID_CAP;
constexpr size_t TD_NA_WORDS = TD_NA_FILL + TD_FILL_WORDS;          // 11.75 MB
static_assert(CT_WORDS <= 64, "control words fit their slot");

static __device__ __align__(256) uint32_t scratch[TD_NA_WORDS];

struct TdNoAlloc {
    uint32_t *ptr = nullptr;     // device address of `scratch` on this device
    uint32_t fill_J = 0;         // the J its class masks were built for (0: none)
};
TdNoAlloc g_noalloc[TD_MAX_DEV];
std::mutex g_noalloc_mu;

// Device address of the array on the current device (looked up and the
// decode table built on the first call per device, on stream st).
int td_noalloc_scratch(hipStream_t st, TdScratch *out)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= TD_MAX_DEV) return -1;
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    TdNoAlloc &na = g_noalloc[dev];
    if (!na.ptr) {
        uint32_t *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            fprintf(stderr, "trial_div_launch_kj_noalloc: hipGetSymbolAddress failed: %s\n",
                    hipGetErrorString(e));
            return -1;
        }
        td_rdec_kernel<<<(TD_RDEC_SIZE + 255u) / 256u, 256, 0, st>>>(
            (uint16_t *)(ptr + TD_NA_RDEC));
        if (hipGetLastError() != hipSuccess) return -1;
        na.ptr = ptr;
    }
    *out = TdScratch{};
    out->small = na.ptr + TD_NA_SMALL;
    out->tbl = na.ptr + TD_NA_TBL;
    out->ctrl = na.ptr + TD_NA_CTRL;
    out->rdec = (uint16_t *)(na.ptr + TD_NA_RDEC);
    out->items = na.ptr + TD_NA_ITEMS;
    out->mid = na.ptr + TD_NA_MID;
    out->fill = na.ptr + TD_NA_FILL;
    out->fill_key = &na.fill_J;
    return 0;
}

int td_launch_with(const uint32_t *d_primes, uint32_t n, long long a, long long b, long long c,
                   uint32_t K, uint32_t J, uint32_t *d_bits, hipStream_t st,
                   hipEvent_t ev0, hipEvent_t ev1, TdScratch *s);

int td_launch(const uint32_t *d_primes, uint32_t n, long long a, long long b, long long c,
              uint32_t K, uint32_t J, uint32_t *d_bits, hipStream_t st,
              hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr)
{
    if (K < 1u || J < 1u || K > 9999u || J > 9999u) return -1;
    if (a < 0 || b < 0 || c < 0) return -1;
    if (!d_bits || (n && !d_primes)) return -1;
    TdScratch *s = nullptr;
    if (td_scratch(&s) != 0) return -1;
    return td_launch_with(d_primes, n, a, b, c, K, J, d_bits, st, ev0, ev1, s);
}

int td_launch_with(const uint32_t *d_primes, uint32_t n, long long a, long long b, long long c,
                   uint32_t K, uint32_t J, uint32_t *d_bits, hipStream_t st,
                   hipEvent_t ev0, hipEvent_t ev1, TdScratch *s)
{
    const int dj = J >= 1000u ? 4 : J >= 100u ? 3 : J >= 10u ? 2 : 1;
    td_reset_kernel<<<1, 64, 0, st>>>(s->ctrl);
    // mid-range primes are listed for the split k loop when the j digit
    // groups merge (a - c >= D_j); otherwise td_large_kernel takes them all
    if (n)
        td_split_kernel<<<(n + TD_BLOCK - 1u) / TD_BLOCK, TD_BLOCK, 0, st>>>(
            d_primes, n, s->small, s->mid, a - c >= dj ? TD_LAT_MIN : TD_SMALL_LIMIT, s->ctrl);
    td_small_setup_kernel<<<TD_SETUP_GRID, TD_BLOCK, 0, st>>>(s->small, s->ctrl, a, b, c, s->tbl);
    switch (dj) {
    case 1: td_launch_rest<1>(d_primes, n, a, b, c, K, J, d_bits, *s, st, ev0, ev1); break;
    case 2: td_launch_rest<2>(d_primes, n, a, b, c, K, J, d_bits, *s, st, ev0, ev1); break;
    case 3: td_launch_rest<3>(d_primes, n, a, b, c, K, J, d_bits, *s, st, ev0, ev1); break;
    default: td_launch_rest<4>(d_primes, n, a, b, c, K, J, d_bits, *s, st, ev0, ev1); break;
    }
    if (hipGetLastError() != hipSuccess) {
        if (s->fill_key) *s->fill_key = 0u;      // the class masks may not have been built
        return -1;
    }
    return 0;
}

// Device copy of a host prime list, reused while the caller's list is
// unchanged: same pointer, same count and the same contents, compared word
// for word against a host copy kept from the last upload (no hash, so no
// collision can reuse a stale list).
struct TdPrimeCache {
    const uint32_t *host = nullptr;
    uint32_t count = 0;
    uint32_t *copy = nullptr;    // host copy of the uploaded list
    uint32_t *dev = nullptr;
    size_t cap = 0;
    uint32_t *bits = nullptr;
    size_t bits_cap = 0;
    uint32_t *back = nullptr;    // pinned: the error latch, then a bitmap of up to TD_BACK_WORDS
};

// Bitmaps up to this size (256 KB, 1448 x 1448) pass through pinned memory in
// stream order; for larger ones the extra host copy costs what a blocking copy
// does.
constexpr size_t TD_BACK_WORDS = 1u << 16;

TdPrimeCache g_cache[TD_MAX_DEV];

// a[0..n) == b[0..n).  The full list below 10^8 is 23 MB, which one core
// reads in about 3 ms, so lists above 4 MB are split over up to 8 threads.
bool td_same_words(const uint32_t *a, const uint32_t *b, uint32_t n)
{
    const size_t bytes = (size_t)n * sizeof(uint32_t);
    if (bytes < ((size_t)4 << 20)) return memcmp(a, b, bytes) == 0;
    unsigned nt = std::thread::hardware_concurrency();
    nt = nt < 2u ? 2u : nt > 8u ? 8u : nt;
    const size_t per = (n + nt - 1u) / nt;
    std::atomic<bool> differ{false};
    auto part = [&](unsigned t) {
        const size_t lo = (size_t)t * per, hi = std::min((size_t)n, lo + per);
        if (lo < hi && memcmp(a + lo, b + lo, (hi - lo) * sizeof(uint32_t)) != 0)
            differ.store(true, std::memory_order_relaxed);
    };
    std::vector<std::thread> th;
    try {
        for (unsigned t = 1; t < nt; t++) th.emplace_back(part, t);
    } catch (...) {
        for (auto &x : th) x.join();
        return memcmp(a, b, bytes) == 0;
    }
    part(0);
    for (auto &x : th) x.join();
    return !differ.load();
}

double td_secs(hipEvent_t x, hipEvent_t y)
{
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, x, y);
    return (double)ms * 1e-3;
}

// Read and clear the error latch of one control block (device memory).
int td_take_error(uint32_t *ctrl)
{
    uint32_t err = 0;
    if (hipMemcpy(&err, ctrl + CT_ERROR, sizeof(err), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    if (err) {
        const uint32_t zero = 0;
        if (hipMemcpy(ctrl + CT_ERROR, &zero, sizeof(zero), hipMemcpyHostToDevice) != hipSuccess)
            return -1;
    }
    return (int)err;
}

int td_check_error_code()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= TD_MAX_DEV) return -1;
    TdScratch &s = g_scratch[dev];
    return s.ready ? td_take_error(s.ctrl) : 0;
}

// The allocation-free launches' latch on the current device.
int td_check_error_noalloc()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= TD_MAX_DEV) return -1;
    uint32_t *ptr = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_noalloc_mu);
        ptr = g_noalloc[dev].ptr;
    }
    return ptr ? td_take_error(ptr + TD_NA_CTRL) : 0;
}

int td_run_host(const prime_list_t *pl, long long a, long long b, long long c,
                uint32_t K, uint32_t J, uint32_t *bits, size_t n_words,
                gpu_timing_t *timing, const char *who)
{
    hipEvent_t e0 = nullptr, e1 = nullptr, e2 = nullptr, e3 = nullptr;
    int dev = 0;
    int rc = -1;
    const size_t need = ((size_t)K * J + 31u) / 32u;
    const size_t bb = need * sizeof(uint32_t);
    TdPrimeCache *pc = nullptr;
    bool fresh = false;
    const bool pinned = need <= TD_BACK_WORDS;
    if (timing) *timing = gpu_timing_t{0.0, 0.0, 0.0};
    if (!pl || !bits || n_words < need || K < 1u || J < 1u || K > 9999u || J > 9999u ||
        a < 0 || b < 0 || c < 0 || (pl->count && !pl->primes)) {
        fprintf(stderr, "%s: invalid arguments\n", who);
        return -1;
    }
    PF_TRY(who, hipGetDevice(&dev));
    if (dev < 0 || dev >= TD_MAX_DEV) goto fail;
    pc = &g_cache[dev];
    if (!pc->back)
        PF_TRY(who, hipHostMalloc(&pc->back, (1 + TD_BACK_WORDS) * sizeof(uint32_t), hipHostMallocDefault));
    PF_TRY(who, hipEventCreate(&e0));
    PF_TRY(who, hipEventCreate(&e1));
    PF_TRY(who, hipEventCreate(&e2));
    PF_TRY(who, hipEventCreate(&e3));
    {
        // Same pointer and count as the cached list: launch on the device
        // copy at once and compare the contents on the host while the
        // kernels run; if they differ, that run is dropped and the call
        // runs again on a fresh upload.
        bool speculative = pc->dev && pc->host == pl->primes && pc->count == pl->count &&
                           pc->bits_cap >= need;
        if (speculative) {
            PF_TRY(who, hipEventRecord(e0, nullptr));
            if (pinned) {
                memcpy(pc->back + 1, bits, bb);
                PF_TRY(who, hipMemcpyAsync(pc->bits, pc->back + 1, bb, hipMemcpyHostToDevice, nullptr));
            } else {
                PF_TRY(who, hipMemcpy(pc->bits, bits, bb, hipMemcpyHostToDevice));
            }
            PF_TRY(who, hipEventRecord(e1, nullptr));
            if (td_launch(pc->dev, pl->count, a, b, c, K, J, pc->bits, nullptr) != 0) {
                fprintf(stderr, "%s: HIP error (kernel launch)\n", who);
                goto fail;
            }
            if (pl->count && !td_same_words(pc->copy, pl->primes, pl->count)) {
                PF_TRY(who, hipDeviceSynchronize());     // the run on the stale list ends unused
                (void)td_check_error_code();
                speculative = false;
            }
        }
        fresh = !speculative;
        if (fresh) {
            pc->host = nullptr;  // invalid until the copy below succeeds
            if (pc->cap < pl->count) {
                if (pc->dev) PF_TRY(who, hipFree(pc->dev));
                free(pc->copy);
                pc->dev = nullptr;
                pc->copy = nullptr;
                pc->cap = 0;
                PF_TRY(who, hipMalloc(&pc->dev, (size_t)pl->count * sizeof(uint32_t) + 4));
                pc->copy = (uint32_t *)malloc((size_t)pl->count * sizeof(uint32_t) + 4);
                if (!pc->copy) {
                    fprintf(stderr, "%s: out of host memory\n", who);
                    goto fail;
                }
                pc->cap = pl->count;
            }
            if (!pc->dev) PF_TRY(who, hipMalloc(&pc->dev, 4));
            if (pc->bits_cap < need) {
                if (pc->bits) PF_TRY(who, hipFree(pc->bits));
                pc->bits = nullptr;
                pc->bits_cap = 0;
                PF_TRY(who, hipMalloc(&pc->bits, bb));
                pc->bits_cap = need;
            }
            PF_TRY(who, hipEventRecord(e0, nullptr));
            if (pl->count)
                PF_TRY(who, hipMemcpy(pc->dev, pl->primes, (size_t)pl->count * sizeof(uint32_t),
                                      hipMemcpyHostToDevice));
            PF_TRY(who, hipMemcpy(pc->bits, bits, bb, hipMemcpyHostToDevice));
            if (pl->count) memcpy(pc->copy, pl->primes, (size_t)pl->count * sizeof(uint32_t));
            pc->host = pl->primes;
            pc->count = pl->count;
            PF_TRY(who, hipEventRecord(e1, nullptr));
            if (td_launch(pc->dev, pl->count, a, b, c, K, J, pc->bits, nullptr) != 0) {
                fprintf(stderr, "%s: HIP error (kernel launch)\n", who);
                goto fail;
            }
        }
        // The error latch and the bitmap come back behind the kernels, and the
        // host waits once: 340 -> 312 us a call at 100 x 100 and the primes below
        // 10^8, against a wait for the kernels and blocking copies.
        PF_TRY(who, hipEventRecord(e2, nullptr));
        PF_TRY(who, hipMemcpyAsync(pc->back, g_scratch[dev].ctrl + CT_ERROR, sizeof(uint32_t),
                                   hipMemcpyDeviceToHost, nullptr));
        if (pinned)
            PF_TRY(who, hipMemcpyAsync(pc->back + 1, pc->bits, bb, hipMemcpyDeviceToHost, nullptr));
        PF_TRY(who, hipEventRecord(e3, nullptr));
        PF_TRY(who, hipEventSynchronize(e3));
        const int err = pc->back[0] ? td_check_error_code() : 0;        // (clears the latch)
        if (err != 0) {
            fprintf(stderr, "%s: %s\n", who,
                    (err & 1) ? "prime outside [2, 2^31) in list"
                    : (err & 2) ? "more than 65536 list entries below 2^16"
                    : (err & 4) ? "more than 1100000 list entries from 2^16 to the lattice range"
                                : "HIP error (error flag readback)");
            goto fail;
        }
        if (pinned) {
            memcpy(bits, pc->back + 1, bb);
        } else {
            PF_TRY(who, hipMemcpy(bits, pc->bits, bb, hipMemcpyDeviceToHost));
            PF_TRY(who, hipEventRecord(e3, nullptr));
            PF_TRY(who, hipEventSynchronize(e3));
        }
        if (timing) {
            timing->upload = td_secs(e0, e1);
            timing->kernel = td_secs(e1, e2);
            timing->download = td_secs(e2, e3);
        }
        rc = 0;
    }
fail:
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (e2) (void)hipEventDestroy(e2);
    if (e3) (void)hipEventDestroy(e3);
    return rc;
}

} // namespace

extern "C" int trial_div_gpu(const prime_list_t *pl, long long a, long long b, long long c,
                             uint32_t *sieve_bits, gpu_timing_t *timing)
{
    return td_run_host(pl, a, b, c, 100u, 100u, sieve_bits, KJ_WORDS, timing, "trial_div_gpu");
}

extern "C" int trial_div_gpu_kj(const prime_list_t *pl, long long a, long long b, long long c,
                                uint32_t K, uint32_t J, uint32_t *bits, size_t n_words,
                                gpu_timing_t *timing)
{
    return td_run_host(pl, a, b, c, K, J, bits, n_words, timing, "trial_div_gpu_kj");
}

extern "C" int cuda_get_device_count(void)
{
    int n = 0;
    return hipGetDeviceCount(&n) == hipSuccess ? n : 0;
}

extern "C" int cuda_set_device(int index)
{
    return hipSetDevice(index) == hipSuccess ? 0 : -1;
}

extern "C" int trial_div_launch_kj(const uint32_t *d_primes, uint32_t n_primes,
                                   long long a, long long b, long long c,
                                   uint32_t K, uint32_t J, uint32_t *d_bits, void *stream)
{
    return td_launch(d_primes, n_primes, a, b, c, K, J, d_bits, (hipStream_t)stream);
}

extern "C" int trial_div_launch_kj_ev(const uint32_t *d_primes, uint32_t n_primes,
                                      long long a, long long b, long long c,
                                      uint32_t K, uint32_t J, uint32_t *d_bits, void *stream,
                                      void *ev_lane_start, void *ev_lane_stop)
{
    return td_launch(d_primes, n_primes, a, b, c, K, J, d_bits, (hipStream_t)stream,
                     (hipEvent_t)ev_lane_start, (hipEvent_t)ev_lane_stop);
}

extern "C" int trial_div_check_error(void)
{
    if (hipDeviceSynchronize() != hipSuccess) return -1;
    const int e0 = td_check_error_code();
    const int e1 = td_check_error_noalloc();
    return e0 != 0 ? e0 : e1;
}

extern "C" uint32_t trial_div_lattice_min(void)
{
    return TD_LAT_MIN;
}

extern "C" int trial_div_launch_kj_noalloc(const uint32_t *d_primes, uint32_t n_primes,
                                           long long a, long long b, long long c,
                                           uint32_t K, uint32_t J, uint32_t *d_bits, void *stream)
{
    if (K < 1u || J < 1u || K > 9999u || J > 9999u) {
        fprintf(stderr, "trial_div_launch_kj_noalloc: K = %u, J = %u outside 1..9999 "
                        "(the scratch array is sized for that grid)\n", K, J);
        return -1;
    }
    if (a < 0 || b < 0 || c < 0 || !d_bits || (n_primes && !d_primes)) {
        fprintf(stderr, "trial_div_launch_kj_noalloc: invalid arguments\n");
        return -1;
    }
    const hipStream_t st = (hipStream_t)stream;
    TdScratch s;
    if (td_noalloc_scratch(st, &s) != 0) return -1;
    return td_launch_with(d_primes, n_primes, a, b, c, K, J, d_bits, st, nullptr, nullptr, &s);
}

void trial_div_launch(const uint32_t *d_primes, uint32_t n_primes, uint64_t a, uint64_t b,
                      uint64_t c, uint32_t *d_bits, int block_size)
{
    (void)block_size;
    if (td_launch(d_primes, n_primes, (long long)a, (long long)b, (long long)c, 100u, 100u,
                  d_bits, nullptr) != 0)
        fprintf(stderr, "trial_div_launch: HIP error (kernel launch)\n");
}
