// decode_resident_order.h — which workgroups of the resident decode kernels tell each other what, and why no word is written over before it
// has been read (plain C++: tests/test_resident_order_cpu.py builds the graph of all reads and writes with it).
//
// A word has one place, and its writer puts the next value there without asking.  So whatever a writer waits for in front of the next value
// has to lie behind all reads of the last one.  In a Block, workgroup r of XCD k:
//   q, k, v     put behind x (MLP) of all 32 of the XCD     read by the XCD's workgroups that attend, in front of their x (MLP)
//   partials    put behind q, k, v of the XCD, so as well    read by the XCD's 32, in front of their x (MLP)
//   far sums 1  put behind x (MLP) of the XCD                read by workgroup r of every XCD, in front of its far sums 2
//   x (c_proj)  put behind far sums 1                        read by the XCD's 32, in front of their h
//   h           put behind x (c_proj) of the XCD             read by the XCD's 32, in front of their far sums 2
//   far sums 2  put behind h of the XCD                      read by workgroup r of every XCD, in front of its NEXT far sums 1
//   x (MLP)     put behind far sums 2                        read by the XCD's 32 in front of what they put next
//   picks       put behind the bests of the XCD's 32         read by every workgroup, in front of all it puts in the next step
// Next q, k, v, partials: behind x (MLP) of all readers.  Next far sums 1: behind x (MLP) of this XCD, which is behind far sums 2 of workgroup r
// of every XCD.  Next x (c_proj) of r: its readers' h lie behind those reads, and its own far sums 2 behind their h.  Next h: behind x (MLP), which
// is behind far sums 2 of the XCD, put behind those reads.  Next far sums 2 of r: behind far sums 1 of workgroup r of EVERY XCD, those without
// heads (narrower models than eight heads) among them: these have nothing to add and put zeros, which say that they have read.  (Without them, with fewer heads than XCDs, nothing
// orders an XCD without heads in front of the others: one that was a Block late found its word gone and waited until the call failed.)
// Next x (MLP): behind x (c_proj) of the next Block, put by readers; an XCD without heads: behind far sums 1, 2 as above.  Picks and
// bests: two hand-overs of the next step's first Block lie in between.
//
// What carries the words is gfx950's and not the language's memory model, which gives other workgroups no view of a store of workgroup scope
// (tests/test_resident_words_cpu.py looks at the instructions these become):
//   * a store without sc1 stops in the L2 of its XCD, all of whose compute units share it (their L1s are written through); one with sc1 goes on to
//     the memory side.  A load with sc1 passes the L1.  So a near word is found by its own XCD, a far word by all.
//   * eight aligned bytes are stored and loaded at once: a word's tag and its value belong together, also in 16-byte accesses of two words, each
//     of which has a tag.  No other order between words is assumed: whoever needs two waits for both.
//   * cache rows have no tags.  A wave's vector memory operations are counted in order (vmcnt), and every wave that stores rows polls x (c_proj)
//     behind them, in front of its workgroup's h: when the polled word is there, so are the rows, in this XCD's L2.  They are asked for with
//     sc1, by workgroups of the same XCD, that have waited for h of that Block since (the newest row travels as words).  Between launches the
//     launch boundary does it.
#pragma once

namespace zg {
namespace resident {

constexpr int kXcds = 8, kRanks = 32;
constexpr int kFar1From = kXcds;  // XCDs (0 .. kFar1From - 1) whose workgroups put partial sums of c_proj, and everyone waits for

}  // namespace resident
}  // namespace zg
