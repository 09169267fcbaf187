// Holds a thread up right after each notification of a condition variable, as
// a scheduler may: every thread but the one that g_main names.
#pragma once
#include <dlfcn.h>
#include <pthread.h>
#include <unistd.h>

static pthread_t g_main;

extern "C" int pthread_cond_broadcast(pthread_cond_t *c)
{
   using fn = int (*)(pthread_cond_t *);
   static const fn real = (fn)dlvsym(RTLD_NEXT, "pthread_cond_broadcast", "GLIBC_2.3.2");
   const int rc = real(c);
   if (!pthread_equal(pthread_self(), g_main)) usleep(50000);
   return rc;
}
