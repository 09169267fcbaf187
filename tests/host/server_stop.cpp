// A server destroyed as soon as its last request is done: the worker, held up
// between finishing the request and waiting for the next one, must leave its
// loop.  argv: requests before the end.
#include <cstdio>
#include <cstdlib>

#include "../../include/libGint.h"
#include "slow_notify.hpp"

int main(int argc, char **argv)
{
   g_main = pthread_self();
   void *h = libgint_create_handle();
   libgint_init(h);
   libgint_amd_plan_begin(h);
   libgint_amd_plan_end(h);
   void *srv = libgint_amd_server_create(1024, 1);
   const int n = 10, client = libgint_amd_server_add_client(srv, h, n);
   double P[n] = {}, K[n], t[3];
   for (int r = 0; r < std::atoi(argv[1]); r++) {
      K[0] = 1.0;
      const int64_t id = libgint_amd_server_submit(srv, client, P, K);
      if (id != r || libgint_amd_server_wait(srv, id, t) != 0 || K[0] != 0.0) return 2;
   }
   K[0] = 2.0;
   libgint_amd_server_destroy(srv);
   libgint_amd_destroy_handle(h);
   std::printf("stopped\n");
   return K[0] == 2.0 ? 0 : 3;   // nothing ran after the last request
}
