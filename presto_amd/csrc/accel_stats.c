/*
 * accel_stats.c -- significance of summed powers
 * (src/characteristics.c:389-559) on the host; the formulas are in
 * accel_sigma.h.
 */
#define ACCEL_SIGMA_FN static
#define ACCEL_SIGMA_TOL 1e-16
#include "accel_sigma.h"
#include "presto_accel.h"

/* chi2 with Q(chi2 | 2n) = q */
static double chisq_Qinv_even(double q, int n)
{
    if (q >= 1.0)
        return 0.0;
    double lq = log(q);
    double lo = 0.0, hi = 1.0;
    while (log_chisq_Q(hi, n) > lq)
        hi *= 2.0;
    double x = hi;
    for (int it = 0; it < 200; it++) {
        double g = log_chisq_Q(x, n) - lq;
        if (g > 0.0)
            lo = x;
        else
            hi = x;
        double y = 0.5 * x;
        double dlog = -0.5 * exp((n - 1) * log(y) - lgamma((double) n) - log_head(y, n));
        double xn = x - g / dlog;
        if (!(xn > lo && xn < hi))
            xn = 0.5 * (lo + hi);
        if (fabs(xn - x) <= 1e-15 * x) {
            x = xn;
            break;
        }
        x = xn;
    }
    return x;
}

double accel_candidate_sigma(double power, int numsum, double numtrials)
{
    return sigma_of_power(power, numsum, numtrials);
}

double accel_power_for_sigma(double sigma, int numsum, double numtrials)
{
    double q = exp(log_gauss_Q(sigma)) / numtrials;
    return 0.5 * chisq_Qinv_even(q, numsum);
}
