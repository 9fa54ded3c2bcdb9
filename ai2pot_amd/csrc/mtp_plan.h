// Contraction plan of a linear Moment Tensor Potential level: the reference's tables
// (alpha_index_basic / alpha_index_times / alpha_moment_mapping, parsed from NN.almtp by
// source/descriptor/mtpr/src/mtpParam.cc:82-214) re-ordered on the host for parallel
// execution and kept resident on the device.
//
// The reference executes `times` sequentially: M[dst] += mult * M[m0] * M[m1] in file order
// (include/mtpBasis.h:522-528) and the adjoint sweep in reverse order
// (include/linearMtp.h:295-306).  Here every moment gets a dependency level (basic moments
// are level 0, a product is one above its deepest factor); moments of one level are
// independent, so one lane computes one moment as a gather over its terms:
//   forward : M[dst]  = sum_t mult_t * M[m0_t] * M[m1_t]             levels ascending
//   reverse : adj[m] += sum_t mult_t * adj[dst_t] * M[other_t]       levels descending
// The plan is valid only if no product is read before its last contribution in file order;
// plan creation verifies this.
#pragma once
#include <hip/hip_runtime.h>
#include <vector>

namespace a2p {

constexpr int MTP_SLOT_CAP = 16;
constexpr int MTP_NEST_MAX = 9, MTP_UNITS_MAX = 64, MTP_NO_MOMENT = 0xffff;
// Terms of a slot to a step of the sweeps, and the words of a step: the terms by pairs, 64 lanes each.
constexpr int MTP_DEPTH_STEP = 4, MTP_STEP_WORDS = MTP_DEPTH_STEP / 2 * 64;
// Mark of a control word: a step of a group of leaves (rev_leaf).
constexpr int MTP_CTRL_LEAF = 1 << 29;

// A gather as the wavefronts of a workgroup walk it.  `lists[m]` holds the terms of moment m, in pairs of the same multiplicity
// (one without a partner twice, each time half).  A slot holds up to MTP_SLOT_CAP of them; a longer list is cut into pieces of
// equal length, so that no lane walks a long list alone.  Slots are
// grouped 64 at a time, one to a lane; the pieces of a list lie in one group, a list of up to sixteen within a row of sixteen
// lanes and a longer one from the beginning of a row on, and the wavefront adds their sums (four doubling steps within a row,
// two across).  How long the pieces of a level are is what a wavefront issues for it at least (pack_level); rows are filled
// first fit, deepest lists first.  The words of a group are padded with zero terms to its depth; a word is a pair: x, y = 8 m0 | 8 m1
// << 16 of its terms (byte offsets into an array of doubles), w = upper half of the multiplicity as a double, whose lower half is
// zero, z = slot word in the first word of a step.
// The groups of a level are dealt to the wavefronts, the deepest first and to the one with the least to do, and everything a
// wavefront needs lies in the order in which it needs it: MTP_STEP_WORDS words to a step, and a control word for each step.
// (Lists cut at sixteen terms and laid out in order of length, in steps of four: 244 instead of 229 us for the call at level 20,
// 8192 atoms, 304 instead of 286 for the training step at level 16, 64 structures of 128 atoms.)
struct MtpStream {
    const int4* head;          // [wavefronts] first step, steps, (16 bytes to a load), barriers before the first step
    const int* ctrl;           // MTP_CTRL_LEAF, and at the last step of a group 1 | doubling steps << 1 | barriers to pass << 4
    const int4* words;         // slot word: (moment in the first piece of a list, -1 elsewhere) & 0xffff | pieces of the list behind this one
                               // << 16, plus one
};

struct MtpPlanDevice {
    // sizes
    int n_moms, n_basic, n_times, n_scalar, nmus, kmax;
    int n_levels;              // number of product levels (>= 0)
    // device arrays
    const unsigned* basic;     // [n_basic]    mu | a << 8 | b << 16 | c << 24
    const int* mapping;        // [n_scalar]
    // forward gather (terms of a product: its factors) and reverse gather (terms of a factor: 8 dst | 8 other << 16;
    // sources by level, from the last level to level 0), for workgroups of one wavefront and of four
    MtpStream fwd[2], rev[2];
    // The same for a linear read-out: scalar moments that no product reads (leaves) are left out of the forward gather, and
    // their lists stand with the first sources of the reverse one (control words marked, 8 m0 | 8 m1 << 16).
    MtpStream fwd_core[2], rev_leaf[2];
    const int* mapping_leaf;   // [n_scalar]   mapping | leaf << 16
    // The passes over the neighbours (mtp.hip: tile_products, nested).  ntiles is 0 where the tables do not fit them: a basic moment
    // that occurs twice, a degree beyond MTP_NEST_MAX, more than MTP_UNITS_MAX units.
    // Sums of the basic moments as matrix products: rows (a, b) and columns (mu, c), those with the most moments first, in tiles of
    // 16 x 16, of which only those with a moment are formed.  Lane l supplies row l % 16 and column l % 16 of a tile and receives row
    // 4 v + l / 16 of its column in place v.
    int ntiles;
    const unsigned* tile_ops;              // [ntiles][64] a | b << 5 | mu << 10 | c << 13 of the lane's row and column
    const uint2* tile_place;               // [ntiles][64] basic moments of the lane's four places, 16 bits each (0xffff: none)
    // Sums over the basic moments at one neighbour: for every (mu, c), c downwards, a unit, the polynomial of degree M = deg(mu) - c in x
    // and y whose coefficients are the adjoints, with zeros for moments that the tables leave out.  stream[0]: b downwards, a downwards.
    // stream[1], for two lanes to a neighbour: the moments with a >= b and those with a < b, each in powers of xy downwards and
    // then of x, or of y, downwards (the second half at half_at, with zeros for a = b).
    int nstream[2], half_at;
    const unsigned short* stream_src[2];   // [nstream] basic moment behind a coefficient (0xffff: none)
    // Units dealt to the wavefronts, one or four, in runs of about equal cost: [wavefronts] {units, first coefficient in stream[0] | in
    // stream[1] << 16}, then [wavefronts][64] M | mu << 4 | last of its mu in the run << 7 | c << 8 | share << 13, shares of the mus numbered.
    const int* units[2];
    int nshares[2];                        // shares in all
    unsigned long long mu_shares[2];       // shares of each mu, eight bits each
    // Polynomials of the passes that own a neighbour per lane.  The basic moments (mu, a, b, c) with the same row (a, b) and
    // the same mu are the coefficients of a polynomial in z; its coefficients lie together, highest power first, up to
    // the highest power in the tables (powers the tables leave out: zero).
    int nrows, npoly, ncoef_poly;
    const int* rows;           // [nrows + 1] a | b << 8 | first polynomial << 16, longest rows first
    const int* polys;          // [npoly] mu | length << 4 | first coefficient << 12
    const int* polys_mu;       // [npoly] the same by mu: a | b << 5 | length << 10 | first coefficient << 15
    const int* polys_end;      // [nmus + 1] run of each mu in polys_mu
    const int* poly_pos;       // [n_basic] coefficient of each basic moment
    const unsigned* polys_len; // [npoly] the same, longest first: mu | a << 3 | b << 8 | length << 13 | first coefficient << 18
                               // (null: a coefficient does not fit its field)
    int poly_unique;           // no two basic moments share a coefficient (the usual case: a plain scatter fills them)
    const int* poly_src;       // [ncoef_poly] basic moment behind the coefficient, -1 none, -2 several (poly_off / items)
    const int* poly_off;       // [ncoef_poly+1]
    const int* poly_items;     // [n_basic] basic moments ordered by coefficient
    // The one-hot adjoints of all scalar moments at once (linear-solver components).  A node (s, m) is moment m as an
    // ancestor of scalar moment s: mapping[s] itself, or a factor of a product among its ancestors.  The adjoint
    // sweeps of all read-outs e_s together are one reverse gather over the nodes, laid out like the reverse gather
    // above (a term packs 8 node(dst) | 8 other << 16 with `other` a moment).
    // The basic ancestors of a scalar moment form a list of words node | basic << 16; lists are cut into pieces of equal length,
    // at most MTP_SLOT_CAP words, and placed first fit, deepest first, 64 slots a group, the pieces of a list in neighbouring
    // slots as in the gathers (the wavefront adds their sums, x_bsteps doubling steps).  A group's words are
    // stored interleaved and padded to the group's depth with node x_nodes, whose adjoint is always zero; `basic` is the moment's
    // place among the polynomials' coefficients (poly_pos) when there are as many of them as basic moments (x_polys): word k of
    // slot q is x_bwords[x_bbase[q >> 6] + k * 64 + (q & 63)].
    // The scalar moments are dealt to batches whose nodes fit the kernel's LDS budget (MtpPlan::xbatches); the fields
    // below are those of the batch a launch works on (x_root is -1 for the scalar moments of other batches).
    int x_nodes, x_slots, x_polys;
    const int* x_root;         // [n_scalar] node (s, mapping[s])
    const int* x_seed;         // [x_slots]  scalar moment, in the slot of its list's first piece; -1 elsewhere
    const int* x_brem;         // [x_slots]  pieces of the same list behind this one
    MtpStream x;               // the reverse gather over the nodes, for four wavefronts (a slot word names the node)
    const int* x_bbase;        // [x_slots/64]
    const int* x_bdepth;       // [x_slots/64]
    const int* x_bsteps;       // [x_slots/64]
    const int* x_bwords;
};

// one batch of scalar moments of the components kernel: the x_ fields of MtpPlanDevice
struct MtpXBatch {
    int nodes, slots;
    const int *root, *seed;
    MtpStream x;
    const int *bbase, *bdepth, *bsteps, *brem, *bwords;
};

struct MtpPlan {
    MtpPlanDevice d;
    std::vector<MtpXBatch> xbatches;   // empty: a scalar moment has too many ancestors (components pass by pass)
    void* device_block = nullptr;   // one allocation holding all arrays
    int device = 0;
};

}  // namespace a2p
