// How the tiles of MLA decode's sequences are dealt to runs, one a workgroup. Plain C++:
// the kernels count by wave, a test on the CPU one sequence after the other.
#pragma once

// A workgroup's run: its sequence, the first tile there, and its tiles; how many there are
// to a run of this sequence.
struct Run {
  int seq, at, todo, per;
};

// The least length in [even, most] of a run with which `runs` suffice and each lies in one
// sequence; most + 1: none does. count(n): how many runs of n tiles all sequences take,
// the fewer the longer they are. Most lists are dealt by the first look or by none.
template <class F>
constexpr int least_length(int even, int most, int runs, F count) {
  if (count(even) <= runs) return even;
  if (most == even || count(most) > runs) return most + 1;
  int low = even, high = most;  // too short; enough
  while (high - low > 1) {
    const int mid = (low + high) / 2;
    if (count(mid) <= runs) {
      high = mid;
    } else {
      low = mid;
    }
  }
  return high;
}

// Run `i` of the k that sequence seq's tiles take, of equal length; none may be left for
// the last ones.
template <class D>
constexpr Run run_of_sequence(int seq, int i, int tiles, int k, D div_up) {
  const int per = div_up(tiles, k), at = i * per, left = tiles - at;
  return {seq, at, left < per ? left : per, per};
}

// The run that begins with tile `begin` of the list of all tiles, of which seq's begin
// with `first`; it may go on with the sequences that follow.
constexpr Run run_of_list(int seq, int begin, int first, int per, int total) {
  return {seq, begin - first, total - begin < per ? total - begin : per, per};
}
