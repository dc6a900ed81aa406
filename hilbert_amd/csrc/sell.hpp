// sell.hpp -- SELL-64 gather tables for one sparse operator (A or A^T).
//
// Rows are cut into slices of 64 (one wavefront, one lane per row).  A
// slice stores width(slice) x 64 packed entries, k-major, so that step k of
// all 64 lanes reads 256 contiguous bytes.  An entry is (code << 24) | col:
// col < 2^24 indexes the input vector, code indexes a per-operator table of
// at most 254 distinct coefficients (code 0 = 0.0 is padding).  Rows longer
// than a threshold are stored separately and reduced by a whole wavefront;
// their slice lane carries the marker code 255 at k = 0 and writes nothing.
#pragma once

#include <cstdint>
#include <vector>

#include "constraints.hpp"

namespace v2h {

constexpr uint32_t kCodeLongRow = 255;

struct SellHost {
    int64_t nrows = 0;
    int nslices = 0;
    std::vector<uint32_t> slice_start;  // [nslices + 1], in units of 64 entries
    std::vector<uint32_t> ent;
    std::vector<int32_t> long_row;      // [nlong]
    std::vector<uint32_t> long_start;   // [nlong + 1]
    std::vector<uint32_t> long_ent;
    std::vector<double> coef;           // [256]
    int nlong() const { return (int)long_row.size(); }
};

SellHost build_sell(const Csr& M, int long_threshold);

// The same operator cut into pieces of at most kPiece entries of one row, for
// the workgroup that keeps a whole small operator to itself: wide rows would
// leave it waiting for one wavefront.  64 pieces of like length make a slice
// (entries k-major, coefficient codes of S); dst of a piece is its row, or for
// a row of several pieces -1 - position of its partial sum.
constexpr int kPiece = 4;
struct PieceHost {
    std::vector<uint32_t> ent;
    std::vector<uint32_t> slice;   // first entry | width << 28
    std::vector<int32_t> dst;      // [slices][64], kNoPiece where there is none
    std::vector<int32_t> multi;    // rows of several pieces: row, first position, pieces (3 each)
    int nparts = 0;
    int nslices() const { return (int)slice.size(); }
    int nmulti() const { return (int)multi.size() / 3; }
};
constexpr int32_t kNoPiece = INT32_MIN;
PieceHost build_pieces(const Csr& M, const SellHost& S);

}  // namespace v2h
