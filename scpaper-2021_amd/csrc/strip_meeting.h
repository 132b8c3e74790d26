// How the workgroups ("parts") that share a token strip meet at one word, with nothing that depends on two of them being
// resident at once.  The word counts arrivals in bits 0-7, holds a bit for each part that did not wait in bits 8-19, and
// counts the parts that are through in bits 20-31; it is zero before the first arrival and behind the last part.
//
// Whoever arrives last waits for nobody.  The others look at the word a bounded number of times, and then leave their share of
// the projection to the last by their bit.  A part counts itself through in its last touch of the word, so whoever finds
// all the others through is alone with it and clears it.  (The bit and that count may not be one addition: a part that
// finds all there after all goes on, and for as long as its count stood in the word another would take itself for the last.)
//
// Also compiled for the host, where a test steps through every order of the touches.
// `Word`: add(v) adds atomically and returns what was there, clear() stores zero, pause() lets time pass.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define ET_MEET_FN __device__ __forceinline__
#else
#define ET_MEET_FN inline
#endif

namespace et {

constexpr int kMeetMaxParts = 12;
constexpr uint32_t kMeetArrived = 1u, kMeetThrough = 1u << 20;

ET_MEET_FN int meet_here(uint32_t word) { return (int)(word & 255); }

// the last touch of a part
template <class Word> ET_MEET_FN void meet_through(Word word, int parts) {
    if ((int)(word.add(kMeetThrough) >> 20) + 1 == parts) word.clear();
}

// Behind the arrival that found `was`: a mask of the parts whose projection is run here besides this one's, or -1: nothing
// more is to be done.  Unless it is -1, the part ends with meet_through().
template <class Word> ET_MEET_FN int meet_wait(Word word, uint32_t was, int part, int parts, bool projecting, int spin) {
    if (meet_here(was) + 1 == parts) return (int)(was >> 8 & 0xfff);
    if (projecting) {
        for (int n = 0; n < spin; n++) {
            if (meet_here(word.add(0u)) == parts) return 0;
            word.pause();
        }
        // all there after all: the last one did not see the bit, and this share is this part's
        if (meet_here(word.add(1u << (8 + part))) == parts) return 0;
    }  // (a normalisation alone is for the last)
    meet_through(word, parts);
    return -1;
}

}  // namespace et
