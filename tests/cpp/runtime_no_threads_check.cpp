// The host runtime's checks where the system gives no further threads: every call that would have a thread of its own is
// made by the calling thread, with the same streams.
#include <cerrno>
#include <pthread.h>

extern "C" int pthread_create(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*) noexcept { return EAGAIN; }

#define main host_check_main
#include "runtime_host_check.cpp"
#undef main

int main() { return host_check_main(); }
