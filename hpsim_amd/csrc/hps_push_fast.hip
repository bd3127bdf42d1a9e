// hps_push_fast.hip -- the tracking kernels of hps_kernels.hip built a
// second time, with reciprocal division and square roots from v_rsq_f64,
// for batches in the grouped field
// solve (field mode 1, whose field comes from the FP32 product or from the
// surrogate attached to it).
//
// Built with -fapprox-func and -freciprocal-math, an FP64 quotient x / y
// becomes v_rcp_f64(y), two Newton steps, x times the refined reciprocal and
// one FMA correction (7 instructions; the compiler's correctly rounded
// sequence takes 11, the exact build's Quick 9, see hps_math.hpp), and
// quotients by one denominator share its reciprocal (x times the rounded
// 1 / y).  With HPS_FAST_PUSH defined, the square roots of the maps, the kick
// and the deposit (psqrt) come from v_rsq_f64 with one Goldschmidt step and
// one Newton correction (12 instructions instead of 21; Quick 10).  Measured
// on the device, both gave the correctly rounded result for every one of
// 400,000 random quotients and roots between 10^-200 and 10^200.  A zero or
// infinite denominator gives NaN instead of an infinity or zero.  The push
// guards the denominators that can be zero: r and the gap radius on the axis,
// and bgzf <= 0 is a loss.  Every other denominator is a mass, a mesh spacing,
// or a velocity or energy that is positive for any particle still alive.
//
// Against the same file built with correctly rounded quotients and roots and
// the full polynomials (Any, hps_math.hpp; the live-particle push in both),
// static VALU instruction counts of the batched push drop by 12 % (quad class)
// and 17 % (RF-gap class), and by 11 % in the batched deposit.  Four members of
// 2,097,152 particles on 64 x 256: push 251 -> 247 us (quad) and 260 -> 249 us
// (RF gap) a launch, rebuild 96 -> 77.  So the push, bound by its memory
// accesses, gains little by now; the deposit is what the second build pays for.
//
// The batched push of this build visits only the live particles of each
// chunk (segment_body_live in hps_kernels.hip).  It adds each chunk's sums
// in another order than the canonical one.
//
// These modes already differ from the FP64 solve: each member's field comes
// from an FP32 product, within about 1e-6 of the FP64 field.  A last-bit
// change in a division is ten orders of magnitude below that.  Their results
// are held to error bounds against the FP64 oracle, not to its bits.  The
// FP64 field mode and single beams, which are bit-exact against the oracle,
// launch the kernels of hps_kernels.hip as built there.  Index arithmetic
// that takes a quotient (mesh cell, table row) keeps its range checks and
// clamps, so a quotient one unit off at a cell boundary selects a
// neighbouring cell, never an address outside the tables.
#define HPS_FAST_PUSH 1
#include "hps_kernels.hip"
