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
