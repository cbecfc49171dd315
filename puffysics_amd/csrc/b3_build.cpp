/*
 * b3_build.cpp - the identity of this engine build: a digest of its sources
 * (B3_BUILD_ID, from the Makefile).  libb3hover.so reads the engine's own
 * structures where the engine it runs with has the identity that it was
 * compiled with, and keeps to the public calls where it has not.
 */
extern "C" unsigned long long b3i_build_id(void) { return B3_BUILD_ID; }
