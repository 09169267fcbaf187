// Requests of several threads at once: each must get its own number back, also
// when another one submits before it returns.
#include <cstdio>
#include <thread>
#include <vector>

#include "../../include/libGint.h"
#include "slow_notify.hpp"

int main()
{
   g_main = pthread_self();
   void *h = libgint_create_handle();
   libgint_init(h);
   libgint_amd_plan_begin(h);
   libgint_amd_plan_end(h);
   void *srv = libgint_amd_server_create(1024, 1);
   const int n = 10, client = libgint_amd_server_add_client(srv, h, n), threads = 4;
   std::vector<int64_t> ids(threads);
   std::vector<std::thread> t;
   double P[n] = {};
   std::vector<double> K(threads * n);
   for (int i = 0; i < threads; i++)
      t.emplace_back([&, i] {
         double s[3];
         ids[i] = libgint_amd_server_submit(srv, client, P, &K[i * n]);
         libgint_amd_server_wait(srv, ids[i], s);
      });
   for (auto &x : t) x.join();
   int seen = 0;
   for (int64_t id : ids) seen |= 1 << id;
   libgint_amd_server_destroy(srv);
   libgint_amd_destroy_handle(h);
   std::printf("%s\n", seen == (1 << threads) - 1 ? "distinct" : "shared");
   return 0;
}
