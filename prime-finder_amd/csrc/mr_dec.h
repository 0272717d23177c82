// mr_dec.h -- launches of the base-10^13 squaring kernels (mr_dec.hip).
#pragma once
#include "mr_dec_core.h"

namespace mr { namespace dec {

struct Args {
    const int32_t *list;        // launch index -> slot (nullptr: identity)
    const uint8_t *run;         // [n] 1 = the slot squares in this chunk (nullptr: all)
    const Form *form;           // [n]
    const int32_t *path;        // [n] class of the round in progress (0: not here)
    double *dig;                // [n][dstride] digits of the residue
    int dstride;
    const uint32_t *N;          // [n][nstride] modulus, 24-bit limbs (the exponent's bits)
    int nstride;
    int32_t *bitpos;
    const int32_t *sval;
    const uint8_t *alive, *pre;
    const uint32_t *base;
    uint32_t *scr;              // [n][sstride] words; canonical digits go here
    int sstride;
    double *Nt;                 // [n][tstride] transform of N' (DENSE), per prime M words
    double *park;               // [n][pstride] T during a DENSE squaring, then residues (SEQ)
    int tstride, pstride;
};

// A context's Montgomery steps in base 2^43 (Gen): any odd moduli of L limbs.
struct GenArgs {
    Gen g;
    const int32_t *path;        // [n] slots with a class here are not this path's (nullptr: none)
    const uint32_t *N, *one;    // [n][nstride]
    uint32_t *res;              // [n][nstride] 24-bit Montgomery residue (in)
    int nstride;
    const uint32_t *scr;        // [n][sstride] 24-bit limbs of N' mod 2^(24 L) and, half way
    int sstride;                //   up, of R mod N (launch_gen_prepare reads them)
    double *tab;                // [n][5][2 M] transforms of N, N', 2^(24 L) mod N, R mod N,
                                //   an operand
    double *dig;                // [n][dstride] result digits
    int dstride;
    double *park;               // [n][pstride]
    int pstride;
    int32_t *flag;              // [n] set: dig holds a new result
    int32_t *bitpos;
    const int32_t *sval;
    const uint8_t *alive, *pre;
    const uint32_t *base;
};
void launch_gen_prepare(const GenArgs &A, const double *tab, int n, hipStream_t st);
// Up to `steps` exponent bits of every slot with a base of at most MAX_BASE; the
// residue's digits (24-bit Montgomery form) to dig.
void launch_gen_exp(const GenArgs &A, const double *tab, int n, int steps, hipStream_t st);
// dig = a b 2^(-24 L) mod N (b == nullptr: a^2) for 24-bit limbs, one per uint64_t.
void launch_gen_mul(const GenArgs &A, const double *tab, int n, const uint64_t *a, const uint64_t *b, int ld,
                    hipStream_t st);

// The class's twiddle tables on the current device (built once per device,
// kept): [prime][forward, inverse].  nullptr on an error.
const double *tables(int device, int lm);
// Up to `steps` exponent bits of every listed slot whose round runs in class lm.
void launch_exp(int lm, const Args &A, const double *tab, int n, int steps, hipStream_t st);
// The transform of N' of the listed slots of class lm that are DENSE.
void launch_prepare(int lm, const Args &A, const double *tab, int n, hipStream_t st);
// a^d mod N's (or the residue in progress's) canonical digits, in [0, 1.1 N),
// as Lw doubles at scr.
void launch_norm(int lm, const Args &A, int n, hipStream_t st);
// form[slot] from terms ([n][2 nterm] by launch index) and the host's choice
// ([n][3]: D, class, mode); a form that does not come out as chosen sets bit 2
// (value 4) of *err.
void launch_form(const int32_t *list, int n, const int64_t *terms, int nterm, const int32_t *choice,
                 Form *form, uint32_t *err, hipStream_t st);

} } // namespace mr::dec
