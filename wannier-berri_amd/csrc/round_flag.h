// "Some pair of this round rotates": a flag of wave 0 to every wave of its workgroup, two LDS words in turn.
#pragma once

#ifdef __HIPCC__
#define WBMI_ROUND_FN __device__ inline
#else
#define WBMI_ROUND_FN inline
#endif

// Wave 0 puts a round's flag, a barrier follows, every wave takes it.  A round that rotates nothing has no other
// barrier, so wave 0 may put the next round's flag before a late wave has taken this one's: it goes to the other word.
// The round after that writes this word again, behind a barrier that every wave reaches only after its take.
// So the words alternate from take to take, whatever sweep a round belongs to (a sweep's number of rounds is
// odd: the parity of the round in its sweep would use one word twice running).
struct RoundFlag {
    int at = 0;
    WBMI_ROUND_FN void put(int* words, int v) const { words[at] = v; }
    WBMI_ROUND_FN int take(const int* words) {
        const int v = words[at];
        at ^= 1;
        return v;
    }
};
